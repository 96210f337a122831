"""Staged 3x3 convolution on images that its 4 x 64-pixel tiles do not divide:
remainders in both directions, one row or pixel, narrow and tiny images, and
the fused pool and head of a prediction at such a size.

Products of bf16 values are exact in float32; the sums are float32, so the
bound is the one of the aligned sizes: 1e-5 of the largest output times the
square root of the input channels, plus 2^-8 of it for the rounded output.
"""
import numpy as np
import pytest

from oracle import unet

pytestmark = pytest.mark.gpu

CASES = [  # n, h, w, c1, up1, c2, cout
    (1, 1, 1, 32, 0, 0, 32),
    (1, 3, 63, 32, 0, 0, 64),
    (2, 5, 65, 64, 0, 0, 32),
    (1, 6, 130, 32, 1, 32, 64),
    (3, 9, 31, 64, 1, 64, 128),
    (1, 130, 8, 32, 0, 0, 96),
    (2, 16, 16, 64, 0, 0, 64),
]


@pytest.mark.parametrize("case", CASES)
def test_convolution_edges(torch_cuda, case):
    torch = torch_cuda
    import cageo_amd.surrogate as sg
    n, h, w, c1, up1, c2, cout = case
    print("CASE conv edges", case, flush=True)
    L, p = sg._nn(), sg._p
    r = np.random.default_rng(sum(case))
    h1, w1 = ((h + 1) // 2, (w + 1) // 2) if up1 else (h, w)
    bits = lambda a: torch.from_numpy((a.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()
    x1 = sg.bf16_round(r.normal(size=(n, h1, w1, c1)).astype(np.float32))
    x2 = sg.bf16_round(r.normal(size=(n, h, w, c2)).astype(np.float32)) if c2 else None
    wt = sg.bf16_round((r.normal(size=(9, cout, c1 + c2)) * 0.1).astype(np.float32))
    b = r.normal(size=cout).astype(np.float32)
    xin = np.repeat(np.repeat(x1, 2, 1), 2, 2)[:, :h, :w] if up1 else x1
    if c2:
        xin = np.concatenate([xin, x2], axis=-1)
    ref = unet.conv3x3(xin.astype(np.float64), wt.astype(np.float64), b)
    d1, dwt, db = bits(x1), bits(wt), torch.from_numpy(b).cuda()
    d2 = bits(x2) if c2 else None
    guard = 64 * cout  # nothing is written past the image
    out = torch.full((n * h * w * cout + guard,), -21846, dtype=torch.int16, device="cuda")
    outf = torch.full((n * h * w * cout + guard,), 7.5, dtype=torch.float32, device="cuda")
    assert L.cageo_nn_conv3x3(None, p(d1), c1, up1, p(d2), c2, p(dwt), p(db), p(out), p(outf), n, h,
                              w, cout, 0) == 0
    only = torch.full((n * h * w * cout + guard,), -21846, dtype=torch.int16, device="cuda")
    assert L.cageo_nn_conv3x3(None, p(d1), c1, up1, p(d2), c2, p(dwt), p(db), p(only), None, n, h, w,
                              cout, 0) == 0
    torch.cuda.synchronize()
    scale = np.abs(ref).max()
    tol = 1e-5 * scale * (c1 + c2) ** 0.5
    assert np.abs(outf[:-guard].cpu().numpy().reshape(ref.shape) - ref).max() <= tol
    u = out[:-guard].cpu().numpy().view(np.uint16).astype(np.uint32) << 16
    assert np.abs(u.view(np.float32).reshape(ref.shape) - ref).max() <= 2.0 ** -8 * scale + tol
    assert torch.equal(out, only)
    assert bool((out[-guard:] == -21846).all()) and bool((outf[-guard:] == 7.5).all())


@pytest.mark.parametrize("shape", [(9, 9), (70, 133), (40, 520)])
def test_prediction_equals_unfused_layers(torch_cuda, shape):
    """A prediction at a ragged size, its pools and head fused, gives the bits
    of the same layers run one by one (the padded width is a multiple of 8)."""
    torch = torch_cuda
    import cageo_amd as ca
    import cageo_amd.surrogate as sg
    print("CASE prediction", shape, flush=True)
    h, w = (s + -s % 8 for s in shape)
    r = np.random.default_rng(h)
    x = np.zeros((1, h, w, sg.IN_PAD), np.float32)
    x[..., :4] = r.normal(size=(1, h, w, 4))
    net = sg.load_net(torch)
    xd = torch.from_numpy(x).cuda()
    ref = net.predict(xd)[0]
    got = torch.empty((h, w), dtype=torch.float32, device="cuda")
    xb = torch.from_numpy((sg.bf16_round(x).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()
    with ca.Surrogate(sg.DEFAULT_WEIGHTS, torch.cuda.current_stream()) as s:
        s.forward(xb, h, w, got)
        torch.cuda.synchronize()
    assert torch.equal(got, ref)
