"""A trainer of a base that does not train holds and saves its weights; its
gradient, step and train calls are refused before they take the batch's
workspace or run anything.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("base", [64, 96, 128])
def test_other_bases_are_refused_at_once(torch_cuda, tmp_path, base):
    torch = torch_cuda
    import cageo_amd as ca
    from cageo_amd import surrogate as sg
    print("CASE trainer base", base, flush=True)
    x = torch.zeros((4, 256, 256, 4), dtype=torch.float32, device="cuda")
    y = torch.zeros((4, 256, 256), dtype=torch.float32, device="cuda")
    with ca.Trainer(base, seed=1, stream=torch.cuda.current_stream()) as tr:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for call in (lambda: tr.gradients(x, y), lambda: tr.step(x, y, 1e-3),
                     lambda: tr.train(x, y, 2, 1e-3, 0.1, 0, 1, 1, 7)):
            with pytest.raises(ca.CageoError) as err:
                call()
            assert err.value.status == -1
        torch.cuda.synchronize()
        # (the workspace of four tiles of 256^2 takes 365 MB and more)
        assert torch.cuda.mem_get_info()[0] >= free - (64 << 20)
        path = str(tmp_path / "w.bin")
        tr.save(path)
    assert sg.load_params(path)["enc1b.w"].shape == (9, base, base)
