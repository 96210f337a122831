"""Weight gradient of the 3x3 convolution at the edges of its tiles: 64-pixel
segments with a remainder, odd numbers of rows, one row, several rounds of the
row ring, both channel block sizes and inputs read at half resolution.

The products of bf16 values are exact in float32 and the sums are float32, so
the error is the summation's: at most the number of summed pixels times
2^-24 of the sum of magnitudes, and of the order of its square root times
2^-24 in practice; the bound is 2^-22 x sqrt(pixels) of the largest sum of
magnitudes.
"""
import numpy as np
import pytest

from oracle import unet

pytestmark = pytest.mark.gpu

CASES = [  # n, h, w, c1, up1, c2, cout
    (1, 1, 1, 32, 0, 0, 32),
    (1, 1, 64, 32, 0, 0, 64),
    (1, 2, 63, 32, 0, 0, 32),
    (2, 5, 65, 64, 0, 0, 64),
    (1, 7, 130, 32, 0, 32, 96),
    (1, 37, 64, 32, 0, 0, 32),
    (3, 10, 33, 64, 1, 32, 64),
    (1, 11, 67, 32, 1, 64, 32),
    (1, 4, 128, 128, 0, 0, 128),
]


@pytest.mark.parametrize("case", CASES)
def test_weight_gradient_edges(torch_cuda, case):
    torch = torch_cuda
    import cageo_amd.surrogate as sg
    n, h, w, c1, up1, c2, cout = case
    print("CASE wgrad", case, flush=True)
    L, p = sg._nn(), sg._p
    r = np.random.default_rng(sum(case))
    h1, w1 = ((h + 1) // 2, (w + 1) // 2) if up1 else (h, w)
    bits = lambda a: torch.from_numpy((a.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()
    x1 = sg.bf16_round(r.normal(size=(n, h1, w1, c1)).astype(np.float32))
    x2 = sg.bf16_round(r.normal(size=(n, h, w, c2)).astype(np.float32)) if c2 else None
    g = sg.bf16_round(r.normal(size=(n, h, w, cout)).astype(np.float32))
    xin = np.repeat(np.repeat(x1, 2, 1), 2, 2)[:, :h, :w] if up1 else x1
    if c2:
        xin = np.concatenate([xin, x2], axis=-1)
    wt = np.zeros((9, cout, c1 + c2))
    _, ref, _ = unet.conv3x3_back(xin.astype(np.float64), wt, g.astype(np.float64))
    _, mag, _ = unet.conv3x3_back(np.abs(xin).astype(np.float64), wt, np.abs(g).astype(np.float64))
    d1, dg = bits(x1), bits(g)
    d2 = bits(x2) if c2 else None
    dw = torch.ones((9, cout, c1 + c2), dtype=torch.float32, device="cuda")  # added to
    assert L.cageo_nn_conv3x3_wgrad(None, p(d1), c1, up1, p(d2), c2, p(dg), p(dw), n, h, w, cout) == 0
    torch.cuda.synchronize()
    bound = 2.0 ** -22 * (n * h * w) ** 0.5 * (mag.max() + 1.0)
    assert np.abs(dw.cpu().numpy() - 1.0 - ref).max() <= bound
