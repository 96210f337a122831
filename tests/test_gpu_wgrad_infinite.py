"""Weight gradient of the 3x3 convolution where an input is infinite at the
image's edge: a tap that moves that pixel out of the image has no product with
it, so its gradient stays finite.  The pixels beyond the edge and the row
below the last are padding of the kernel's 64-pixel segments and row pairs.

The bound of the finite gradients is the one of the other sizes: 2^-22 x
sqrt(pixels) of the largest sum of magnitudes.
"""
import numpy as np
import pytest

from oracle import unet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(1, 1), (5, 30), (7, 33), (6, 63), (3, 64), (9, 95), (4, 97), (5, 130)])
@pytest.mark.parametrize("cout", [32, 64])
def test_infinite_pixels_at_the_edges(torch_cuda, h, w, cout):
    torch = torch_cuda
    import cageo_amd.surrogate as sg
    print("CASE wgrad infinite", h, w, cout, flush=True)
    L, p = sg._nn(), sg._p
    r = np.random.default_rng(100 * h + w)
    x = sg.bf16_round(r.normal(size=(1, h, w, 32)).astype(np.float32))
    g = sg.bf16_round((r.normal(size=(1, h, w, cout)) + 0.001).astype(np.float32))
    g[g == 0] = 1.0
    finite = x.copy()
    edges = ((0, 0), (0, w - 1), (h - 1, 0), (h - 1, w - 1), (h // 2, w - 1), (h - 1, w // 2))
    for k, (y, xx) in enumerate(edges):  # one channel each
        x[0, y, xx, 5 * k] = np.inf
        finite[0, y, xx, 5 * k] = 0.0
    wt = np.zeros((9, cout, 32))
    _, ref, _ = unet.conv3x3_back(finite.astype(np.float64), wt, g.astype(np.float64))
    _, mag, _ = unet.conv3x3_back(np.abs(finite).astype(np.float64), wt, np.abs(g).astype(np.float64))
    for k, (y, xx) in enumerate(edges):
        for tap in range(9):
            gy, gx = y - (tap // 3 - 1), xx - (tap % 3 - 1)
            if 0 <= gy < h and 0 <= gx < w:
                ref[tap, :, 5 * k] = np.inf * g[0, gy, gx]
    bits = lambda a: torch.from_numpy((a.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()
    dx, dg = bits(x), bits(g)
    dw = torch.zeros((9, cout, 32), dtype=torch.float32, device="cuda")
    assert L.cageo_nn_conv3x3_wgrad(None, p(dx), 32, 0, None, 0, p(dg), p(dw), 1, h, w, cout) == 0
    torch.cuda.synchronize()
    got = dw.cpu().numpy()
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf].astype(np.float32))
    bound = 2.0 ** -22 * (h * w) ** 0.5 * (mag.max() + 1.0)
    assert np.abs(got[~inf] - ref[~inf]).max() <= bound
