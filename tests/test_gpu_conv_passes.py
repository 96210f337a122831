"""The Gaussian convolution's two passes where their steps and wraps end: taps
at and past a multiple of 16, halos at the widths where the rows pass changes
its layout (r = 16, 17, 32, 33), rasters narrower than a tile and its halo
(an index wraps more than once) and ragged ones.  The order of the sums is the
oracle's, so the results are equal bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [0, 1, 7, 8, 15, 16, 17, 32, 33, 60])
@pytest.mark.parametrize("h,w", [(1, 1), (5, 200), (79, 80), (64, 128), (97, 161), (200, 33)])
def test_passes_bit_exact(torch_cuda, h, w, r):
    import cageo_amd as ca

    if r > min(h, w):
        pytest.skip("a radius beyond the raster is refused")
    print("CASE conv passes", h, w, r, flush=True)
    torch = torch_cuda
    g = np.random.default_rng(1000 * h + 10 * w + r)
    z = g.standard_normal((h, w)).astype(np.float32)
    f = g.uniform(-0.2, 1.0, 2 * r + 1).astype(np.float32)
    with ca.Context(w, h, torch.cuda.current_stream()) as ctx:
        ctx.set_filter(ca.GAUSSIAN, r, f)
        t = torch.from_numpy(z).cuda()
        ctx.convolve(t)
        got = t.cpu().numpy()
    assert np.array_equal(got, oracle.convolve(z, f, r, oracle.GAUSSIAN))
