"""Flow tracing where the chains between tiles can go wrong: one path through
every cell of a grid (thousands of exits one after the other), cycles through
several tiles with paths that lead into them, and grids at the edges of a
tile.  Whole numbers: equal to the oracle's."""
import numpy as np
import pytest

import oracle
from helpers import NODATA

pytestmark = pytest.mark.gpu


def announce(*what):
    print("CASE", *what, flush=True)


@pytest.fixture(scope="module")
def ca(torch_cuda):
    import cageo_amd

    return cageo_amd


def trace(ca, torch, fd, stream, workgroups=0):
    h, w = stream.shape
    with ca.Context(w, h, torch.cuda.current_stream()) as ctx:
        if workgroups:
            ctx.configure(workgroups, 0)
        lab = torch.empty((h, w), dtype=torch.int32, device="cuda")
        args = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (fd, stream)]
        longp = ctx.flow_tracing(lab, *args)
        first = lab.cpu().numpy()
        assert ctx.flow_tracing(lab, *args) == longp  # again, over the buffers the first left
        assert np.array_equal(lab.cpu().numpy(), first)
    ref = oracle.flow_tracing(fd, stream)
    assert np.array_equal(first, ref), int((first != ref).sum())
    return longp


def snake(h, w, down):
    """Directions of one path through every cell: along the rows (`down`: in
    bands of one row going down), boustrophedon, out of the grid at its end."""
    fd = np.zeros((h, w, 2), np.int8)
    for y in range(h):
        right = y % 2 == 0
        fd[y, :, 0] = 1 if right else -1
        end = w - 1 if right else 0
        fd[y, end] = (0, 1)
    return fd if down else np.ascontiguousarray(fd[::-1, ::-1] * np.int8(-1))


@pytest.mark.parametrize("workgroups", [0, 1, 3])
@pytest.mark.parametrize("h,w,down", [(65, 63, True), (200, 321, False), (300, 301, True)])
def test_one_path(ca, torch_cuda, h, w, down, workgroups):
    announce("path", h, w, down, workgroups)
    stream = np.full((h, w), NODATA, np.float32)
    fd = snake(h, w, down)
    assert trace(ca, torch_cuda, fd, stream, workgroups) == 0
    stream[h // 2, w // 3] = 3.0  # cells above reach it, cells below leave the grid
    assert trace(ca, torch_cuda, fd, stream, workgroups) == 0


@pytest.mark.parametrize("side", [2, 63, 64, 65, 150])
def test_cycles(ca, torch_cuda, side):
    """A square ring of cells that lead round, and a row above it into it."""
    announce("cycle", side)
    h, w = 211, 260
    y0, x0 = 1, 50
    fd = np.zeros((h, w, 2), np.int8)
    fd[..., 1] = 1  # out of the grid
    y1, x1 = y0 + side - 1, x0 + side - 1
    fd[y0, x0:x1] = (1, 0)
    fd[y0:y1, x1] = (0, 1)
    fd[y1, x0 + 1:x1 + 1] = (-1, 0)
    fd[y0 + 1:y1 + 1, x0] = (0, -1)
    stream = np.full((h, w), NODATA, np.float32)
    stream[y0 + 1:y1, x0 + 1:x1] = 2.0
    trace(ca, torch_cuda, fd, stream)
    stream[y1, (x0 + x1) // 2] = 5.0  # opens the ring
    trace(ca, torch_cuda, fd, stream)
