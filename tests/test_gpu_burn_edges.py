"""Stream burning at the edges of its 64 x 32 blocks and 8-row waves: every
bevel radius, streams few and many, cells of no data on and off the streams,
and no data equal to a burned cell's 0.  Equal to the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodata", [-9999.0, 0.0])
@pytest.mark.parametrize("h,w", [(1, 1), (8, 64), (31, 63), (33, 65), (64, 128), (97, 130)])
def test_burn_edges(torch_cuda, h, w, nodata):
    import cageo_amd as ca

    torch = torch_cuda
    r = np.random.default_rng(h * 1000 + w)
    for bevel in range(ca.MAX_BEVEL_RADIUS + 1 if hasattr(ca, "MAX_BEVEL_RADIUS") else 6):
        for share in (0.004, 0.08, 0.6):
            print("CASE burn", h, w, nodata, bevel, share, flush=True)
            z = r.uniform(0.5, 900.0, (h, w)).astype(np.float32)
            z[r.random((h, w)) < 0.1] = nodata
            stream = np.full((h, w), -1.0, np.float32)
            on = r.random((h, w)) < share
            stream[on] = r.integers(0, 9, int(on.sum())).astype(np.float32)
            with ca.Context(w, h, torch.cuda.current_stream()) as ctx:
                tz = torch.from_numpy(z).cuda()
                ctx.stream_burn(tz, torch.from_numpy(stream).cuda(), bevel, nodata, -1.0)
                got = tz.cpu().numpy()
            ref = oracle.stream_burn(z, stream, bevel, nodata, -1.0)
            assert np.array_equal(got, ref), int((got != ref).sum())
