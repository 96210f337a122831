"""The pit fill's two bounds against the oracle, bit for bit, where they
differ most and where tiles leave a workgroup's LDS.

Grids made of dead levels (values that fail the reference's bucket round
trip) keep many cells undecided, so several lower and upper bounds are taken;
a launch with fewer workgroups than tiles reloads tiles between visits,
takes blocks in turn and hands the last lower bound over.  Equality with the
oracle is exact: the result is unique.
"""
import numpy as np
import pytest

import oracle
from helpers import NODATA, mm_grid, rng, synth_case

pytestmark = pytest.mark.gpu


def announce(*what):
    print("CASE", *what, flush=True)


def dead_levels(mn, hi):
    """Whole millimetres below `hi` whose elevation fails the round trip with
    the raster's minimum `mn` (float32, as the reference evaluates it)."""
    v = (np.arange(1, hi) / np.float32(1000.0)).astype(np.float32)
    mn = np.float32(mn)
    idx = (np.float32(1000.0) * (v - mn)).astype(np.uint64)
    back = (idx.astype(np.float32) / np.float32(1000.0) + mn).astype(np.float32)
    return v[back != v], v[back == v]


def grid(kind, r, h, w):
    if kind == "half_dead":
        dead, live = dead_levels(0.0, 4000)
        z = np.where(r.random((h, w)) < 0.5, r.choice(dead, (h, w)), r.choice(live, (h, w)))
        z[r.random((h, w)) < 0.002] = 0.0  # the raster's minimum, and seeds
        return z.astype(np.float32)
    if kind == "nodata":  # the nodata value is the minimum: most levels are dead
        z = mm_grid(r, h, w, 1, 3000, 0.002)
        z[r.random((h, w)) < 0.01] = NODATA
        z[h // 4:h // 3, w // 5:w // 2] = NODATA
        return z
    if kind == "walled":  # an inner part nothing reaches: it keeps Z
        z = mm_grid(r, h, w, 1, 900, 0.0)
        z[h // 4:h // 4 + 3, w // 4:3 * w // 4] = NODATA
        z[3 * h // 4:3 * h // 4 + 3, w // 4:3 * w // 4 + 3] = NODATA
        z[h // 4:3 * h // 4 + 3, w // 4:w // 4 + 3] = NODATA
        z[h // 4:3 * h // 4 + 3, 3 * w // 4:3 * w // 4 + 3] = NODATA
        return z
    dem, stream = synth_case(max(h, w), seed=3)
    return oracle.stream_burn(dem[:h, :w].copy(), stream[:h, :w].copy(), 2, NODATA, NODATA)


@pytest.mark.parametrize("workgroups", [0, 1, 3, 7])
@pytest.mark.parametrize("kind,shape", [("half_dead", (130, 257)), ("half_dead", (65, 64)),
                                        ("nodata", (200, 193)), ("walled", (260, 140)),
                                        ("synth", (320, 450))])
def test_pit_fill_bounds(torch_cuda, kind, shape, workgroups):
    import cageo_amd as ca
    torch = torch_cuda
    announce("pit_fill bounds", kind, shape, workgroups)
    h, w = shape
    z = grid(kind, rng(70 + h), h, w)
    ref, qref = oracle.pit_fill(z, float(NODATA))
    with ca.Context(w, h) as ctx:
        ctx.configure(workgroups)
        d = torch.from_numpy(z.copy()).cuda()
        filled = torch.empty_like(d)
        for _ in range(2):  # the second call meets the first one's workspace
            ctx.pit_fill(filled, d, float(NODATA))
            assert np.array_equal(d.cpu().numpy(), qref)
            got = filled.cpu().numpy()
            assert np.array_equal(got, ref), f"{(got != ref).sum()} cells differ"
            d.copy_(torch.from_numpy(z))
