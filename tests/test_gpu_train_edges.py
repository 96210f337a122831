"""Fused backward passes of the trainer at sizes that the convolution's tiles
do not divide at some level: its gradients against the same network run layer
by layer (whose kernels the float64 oracle checks).

Both round the same float32 values to bf16 at the same places, so they
differ by the order of float32 sums, and where such a difference crosses a
bf16 rounding boundary by 2^-8 of one of many summed values: 2e-3 of a
tensor's largest gradient, the bound of the aligned size.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w", [(1, 8, 8), (3, 24, 40), (2, 64, 72), (1, 200, 136)])
def test_trainer_gradients_ragged(torch_cuda, tmp_path, n, h, w):
    torch = torch_cuda
    import cageo_amd as ca
    from cageo_amd import surrogate as sg
    print("CASE trainer gradients", n, h, w, flush=True)
    path = str(tmp_path / "init.bin")
    sg.save_params(sg.init_params(32, seed=5), path)
    net = sg.UNet(torch, base=32, params=sg.load_params(path))
    rng = np.random.default_rng(n * h + w)
    x = np.zeros((n, h, w, sg.IN_PAD), np.float32)
    x[..., 0] = rng.normal(0.0, 1.0, (n, h, w))
    x[..., 1] = rng.random((n, h, w)) < 0.1
    x[..., 2:4] = 0.6
    y = torch.from_numpy((rng.random((n, h, w)) * 0.3).astype(np.float32)).cuda()
    net.zero_grad()
    net.forward(torch.from_numpy(x).cuda())
    loss = net.backward(y)
    x4 = torch.from_numpy(np.ascontiguousarray(x[..., :4])).cuda()
    with ca.Trainer(32, init_weights=path, stream=torch.cuda.current_stream()) as tr:
        for _ in range(2):  # the second call replaces the first one's gradients
            got = tr.gradients(x4, y)
            assert abs(got - loss) <= 1e-5 * abs(loss)
            for name, ref in net.grads_numpy().items():
                err = np.abs(tr.read(name, ref.shape, grad=True) - ref).max()
                assert err <= 2e-3 * (np.abs(ref).max() or 1.0), name
