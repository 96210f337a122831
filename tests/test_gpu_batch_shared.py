"""Tiles of a batch that add to one counter raster, wholly or in part: several
error models of one DEM summed into one map.  Every mode gives the sum of the
tiles' own maps, which the per-tile mode computes one after the other.  Each
case prints its name before it touches the GPU.
"""
import pytest

from helpers import NODATA, synth_case

pytestmark = pytest.mark.gpu

H, W = 200, 130
PARAMS = [(1, 60.0, 1.8), (1, 30.0, 0.5), (1, 100.0, 3.0), (0, 60.0, 1.0), (1, 45.0, 2.0),
          (1, 80.0, 1.2)]
N = 4


@pytest.mark.parametrize("rows", [(0, 0, 0, 0, 0, 0),        # one map for all
                                  (0, 0, 200, 0, 400, 400),  # three maps
                                  (0, 100, 199, 299, 500, 600)])  # overlapping ones, out of turn
def test_tiles_that_share_counters(torch_cuda, rows):
    import cageo_amd as ca
    torch = torch_cuda
    print("CASE batch shared counters", rows, flush=True)
    dem, st = synth_case(max(H, W), seed=12)
    dem, st = torch.from_numpy(dem[:H, :W].copy()).cuda(), torch.from_numpy(st[:H, :W].copy()).cuda()

    def maps():
        whole = torch.zeros((max(rows) + H, W), dtype=torch.float32, device="cuda")
        return whole, [whole[r:r + H] for r in rows]

    with ca.Batch([(H, W)] * len(rows)) as b:
        for t, (model, pr, std) in enumerate(PARAMS):
            b.setup_tile(t, dem, st, float(NODATA), float(NODATA), 2, model, pr, 10.0, 0.0, std,
                         77 + t)
        own = [torch.zeros((H, W), dtype=torch.float32, device="cuda") for _ in rows]
        b.run(own, N, first=3, mode=ca.BATCH_PER_TILE)
        ref = maps()[0]
        for r, m in zip(rows, own):
            ref[r:r + H] += m
        assert float(ref.sum()) > 0
        for mode in (ca.BATCH_PER_TILE, ca.BATCH_STREAM, ca.BATCH_GRAPH):
            whole, mcs = maps()
            for _ in range(3):
                whole.zero_()
                b.run(mcs, N, first=3, mode=mode)
                assert torch.equal(whole, ref), mode
