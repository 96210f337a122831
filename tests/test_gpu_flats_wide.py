"""Flats over many tiles whose distances are set and then lowered along whole
rows of a tile, so that rows of many cells, rows of a few and both at once are
compared in a level: constant grids whose last tiles are narrow, plateaus with
walls across the tiles, and both transposed.  Equal to the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(140, 332), (333, 205), (270, 270)])
@pytest.mark.parametrize("form", ["constant", "blocks", "ramps"])
def test_wide_flats(torch_cuda, h, w, form):
    import cageo_amd as ca
    torch = torch_cuda
    print("CASE wide flats", h, w, form, flush=True)
    y, x = np.mgrid[0:h, 0:w]
    z = np.full((h, w), 100.0, np.float32)
    if form == "blocks":
        z[(x % 150 < 100) & (y % 130 < 90)] = 101.0
    if form == "ramps":  # basins of a few levels, each with its outlet in a corner
        z = (100 + (x // 97) + (y // 71)).astype(np.float32)
    for g in (z, np.ascontiguousarray(z.T)):
        gh, gw = g.shape
        with ca.Context(gw, gh, torch.cuda.current_stream()) as ctx:
            fd = torch.empty((gh, gw, 2), dtype=torch.int8, device="cuda")
            ctx.flow_routing(fd, torch.from_numpy(g).cuda())
            assert np.array_equal(fd.cpu().numpy(), oracle.flow_routing(g))
