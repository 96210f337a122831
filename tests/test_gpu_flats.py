"""Flats of the flow routing where the level search of a 64 x 64 tile can go
wrong: grids at the edges of a tile, corridors of more levels than one run
records (255), and lakes fed from several sides of a tile in different passes (a
distance set once and lowered later).  Whole numbers: equal to the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def announce(*what):
    print("CASE", *what, flush=True)


@pytest.fixture(scope="module")
def ca(torch_cuda):
    import cageo_amd

    return cageo_amd


def route(ca, torch, z):
    h, w = z.shape
    with ca.Context(w, h, torch.cuda.current_stream()) as ctx:
        fd = torch.empty((h, w, 2), dtype=torch.int8, device="cuda")
        zd = torch.from_numpy(np.ascontiguousarray(z)).cuda()
        ctx.flow_routing(fd, zd)
        first = fd.cpu().numpy()
        ctx.flow_routing(fd, zd)  # again, over the buffers the first left
        assert np.array_equal(fd.cpu().numpy(), first)
    ref = oracle.flow_routing(z)
    assert np.array_equal(first, ref), int((first != ref).any(-1).sum())


@pytest.mark.parametrize("h,w", [(1, 1), (3, 3), (3, 200), (64, 64), (65, 63), (66, 66), (129, 127)])
def test_plateau_sizes(ca, torch_cuda, h, w):
    announce("flats", h, w)
    r = np.random.default_rng(h * 1000 + w)
    route(ca, torch_cuda, r.integers(1, 3, (h, w)).astype(np.float32))
    route(ca, torch_cuda, np.full((h, w), 7.0, np.float32))


@pytest.mark.parametrize("h,w,step", [(64, 64, 2), (62, 300, 2), (193, 130, 3), (200, 201, 2)])
def test_corridor(ca, torch_cuda, h, w, step):
    """One corridor between walls, `step` rows apart, with its outlet at one end."""
    announce("corridor", h, w, step)
    z = np.full((h, w), 5.0, np.float32)
    rows = list(range(2, h - 2, step))
    for i, y in enumerate(rows):
        z[y, 2:w - 2] = 1.0
        if i + 1 < len(rows):
            z[y:rows[i + 1] + 1, (w - 3) if i % 2 == 0 else 2] = 1.0
    z[rows[-1], w // 2] = 0.5
    for turned in (z, z.T, z[::-1, ::-1]):
        route(ca, torch_cuda, turned)


@pytest.mark.parametrize("seed", range(4))
def test_lakes_across_tiles(ca, torch_cuda, seed):
    """A lake over many tiles, islands in it and a few outlets."""
    announce("lakes", seed)
    r = np.random.default_rng(seed)
    h, w = 260 + 31 * seed, 330 - 17 * seed
    z = np.full((h, w), 2.0, np.float32)
    z[0], z[-1], z[:, 0], z[:, -1] = 9.0, 9.0, 9.0, 9.0
    z[r.random((h, w)) < 0.25] = 3.0
    for _ in range(1 + seed):
        z[r.integers(2, h - 2), r.integers(2, w - 2)] = 1.5
    z[r.integers(2, h - 2), r.integers(2, w - 2)] = 0.0
    route(ca, torch_cuda, z)


@pytest.mark.parametrize("seed", range(3))
def test_drop_ranges(ca, torch_cuda, seed):
    """Drops of every magnitude, denormal to infinite, and diagonal drops about
    the square root of two times the straight ones."""
    announce("drops", seed)
    r = np.random.default_rng(seed)
    h, w = 131, 190
    z = np.float32(10.0) ** r.uniform(-44, 38, (h, w)).astype(np.float32)
    z[r.random((h, w)) < 0.02] = np.inf
    z[r.random((h, w)) < 0.02] = 0.0
    near = np.float32(100.0) - np.float32(0.001) * r.integers(0, 4000, (h, w)).astype(np.float32)
    step = np.where((np.add.outer(np.arange(h), np.arange(w)) & 1) == 0, np.float32(1.0),
                    np.float32(1.4142135))
    ties = (np.float32(7.0) - step * r.integers(0, 2, (h, w)).astype(np.float32) -
            r.integers(0, 3, (h, w)).astype(np.float32) * np.float32(2.0 ** -22))
    with np.errstate(all="ignore"):
        for g in (z, near, ties.astype(np.float32)):
            route(ca, torch_cuda, g)
