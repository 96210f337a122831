"""The 3x3 convolution's two kernels on images that the 4 x 64-pixel tiles do
not divide: batches of narrow images, which the kernel without staging takes,
against float64, and the same images side by side in one wide image, which
the staged kernel takes, against the narrow batch.

Both add the products of tap 0 over all input channels first, then those of
tap 1, and so on, in float32: the same bits whichever kernel a size goes to.
The bound against float64 is the one of the other sizes: 1e-5 of the largest
output times the square root of the input channels, plus 2^-8 of it for the
rounded output.
"""
import numpy as np
import pytest

from oracle import unet

pytestmark = pytest.mark.gpu

N, H, W, PITCH = 54, 37, 8, 10  # 54 x 10 tiles an eighth full: not staged

CASES = [  # c1, up1, c2, cout
    (32, 0, 0, 32),
    (64, 0, 0, 32),
    (32, 0, 32, 64),
    (64, 1, 32, 32),
    (128, 0, 0, 256),
    (128, 1, 64, 64),    # the most channels of a 4-row tile,
    (192, 1, 96, 128),   # of a 2-row one
    (256, 1, 128, 128),  # and of one row
    (256, 0, 0, 64),     # neither kernel stages it
]


@pytest.mark.parametrize("case", CASES)
def test_both_kernels_give_the_same_bits(torch_cuda, case):
    torch = torch_cuda
    import cageo_amd.surrogate as sg
    c1, up1, c2, cout = case
    print("CASE convolution order", case, flush=True)
    L, p = sg._nn(), sg._p
    r = np.random.default_rng(sum(case))
    s = 2 if up1 else 1
    h1, w1 = -(-H // s), W // s
    bits = lambda a: torch.from_numpy((a.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()

    def beside(a, pitch):  # the images side by side, zero pixels between
        n, h, w, c = a.shape
        out = np.zeros((1, h, n, pitch, c), np.float32)
        out[0, :, :, :w] = a.transpose(1, 0, 2, 3)
        return np.ascontiguousarray(out.reshape(1, h, n * pitch, c)[:, :, :n * pitch - (pitch - w)])

    x1 = sg.bf16_round(r.normal(size=(N, h1, w1, c1)).astype(np.float32))
    x2 = sg.bf16_round(r.normal(size=(N, H, W, c2)).astype(np.float32)) if c2 else None
    wt = sg.bf16_round((r.normal(size=(9, cout, c1 + c2)) * 0.1).astype(np.float32))
    b = r.normal(size=cout).astype(np.float32)

    def run(a1, a2, n, w):
        d1, d2 = bits(a1), bits(a2) if c2 else None
        out = torch.empty((n, H, w, cout), dtype=torch.int16, device="cuda")
        outf = torch.empty((n, H, w, cout), dtype=torch.float32, device="cuda")
        only = torch.empty_like(out)
        for o, f in ((out, outf), (only, None)):
            assert L.cageo_nn_conv3x3(None, p(d1), c1, up1, p(d2), c2, p(dw), p(db), p(o), p(f), n, H,
                                      w, cout, 0) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, only)
        return out, outf

    dw, db = bits(wt), torch.from_numpy(b).cuda()
    out, outf = run(x1, x2, N, W)
    wide = N * PITCH - (PITCH - W)
    wout, woutf = run(beside(x1, PITCH // s), beside(x2, PITCH) if c2 else None, 1, wide)

    def apart(a):  # a narrow image's pixels of the wide output
        a = torch.nn.functional.pad(a, (0, 0, 0, PITCH - W))
        return a.view(H, N, PITCH, cout)[:, :, :W].permute(1, 0, 2, 3)

    assert torch.equal(apart(woutf), outf)
    assert torch.equal(apart(wout), out)

    xin = np.repeat(np.repeat(x1, 2, 1), 2, 2)[:, :H, :W] if up1 else x1
    if c2:
        xin = np.concatenate([xin, x2], axis=-1)
    ref = unet.conv3x3(xin.astype(np.float64), wt.astype(np.float64), b)
    scale = np.abs(ref).max()
    tol = 1e-5 * scale * (c1 + c2) ** 0.5
    assert np.abs(outf.cpu().numpy() - ref).max() <= tol
    u = out.cpu().numpy().view(np.uint16).astype(np.uint32) << 16
    assert np.abs(u.view(np.float32) - ref).max() <= 2.0 ** -8 * scale + tol


def test_narrow_prediction_equals_its_layers(torch_cuda):
    """A DEM of one tile's width and some thousand rows, whose full-size
    layers go to the kernel without staging: their pool and head follow by
    themselves, and the prediction has the bits of the layers run one by one."""
    torch = torch_cuda
    import cageo_amd as ca
    import cageo_amd.surrogate as sg
    h, w = 2064, 8
    print("CASE narrow prediction", h, w, flush=True)
    r = np.random.default_rng(8)
    x = np.zeros((1, h, w, sg.IN_PAD), np.float32)
    x[..., :4] = r.normal(size=(1, h, w, 4))
    net = sg.load_net(torch)
    ref = net.predict(torch.from_numpy(x).cuda())[0]
    got = torch.empty((h, w), dtype=torch.float32, device="cuda")
    xb = torch.from_numpy((sg.bf16_round(x).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)).cuda()
    with ca.Surrogate(sg.DEFAULT_WEIGHTS, torch.cuda.current_stream()) as s:
        s.forward(xb, h, w, got)
        torch.cuda.synchronize()
    assert torch.equal(got, ref)
