"""The SGD and Adam kernels' aligned (float4) and element-wise paths, at sizes
around their blocks and remainders and at unaligned addresses, against
torch.optim on the CPU (fp32, the same order of operations: a few ulps of the
update, 1e-6)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 2047, 2048, 2051, 4099, 100001])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("wd", [0.0, 0.01])
def test_sgd_and_adam_match_torch(n, shift, wd):
    from kan_amd import _lib
    print(f"optim n={n} shift={shift} wd={wd}", flush=True)
    lib = _lib.load()
    gen = torch.Generator().manual_seed(n)
    p0, g0 = torch.randn(n, generator=gen), torch.randn(n, generator=gen)
    guard = 8

    def dev(v):  # at byte offset 4 * shift of a 16-byte aligned buffer, guarded on both sides
        buf = torch.full((n + shift + guard,), 7.0, device="cuda")
        buf[shift:shift + n] = v.cuda()
        return buf, buf.data_ptr() + 4 * shift

    pb, pp = dev(p0)
    gb, gp = dev(g0)
    st = _lib.stream_ptr(pb.device)
    _lib.check(lib.ckan_sgd_step(pp, gp, n, 0.1, wd, st))
    ref = p0.clone().requires_grad_(True)
    ref.grad = g0.clone()
    torch.optim.SGD([ref], lr=0.1, weight_decay=wd).step()
    assert torch.allclose(pb[shift:shift + n].cpu(), ref.detach(), rtol=1e-6, atol=1e-6)
    assert torch.all(pb[shift + n:] == 7.0) and torch.all(pb[:shift] == 7.0)

    pb, pp = dev(p0)
    mb, mp = dev(torch.zeros(n))
    vb, vp = dev(torch.zeros(n))
    ref = p0.clone().requires_grad_(True)
    opt = torch.optim.Adam([ref], lr=0.01, weight_decay=wd)
    for step in (1, 2):
        _lib.check(lib.ckan_adam_step(pp, gp, mp, vp, n, step, 0.01, 0.9, 0.999, 1e-8, wd, st))
        ref.grad = g0.clone()
        opt.step()
    assert torch.allclose(pb[shift:shift + n].cpu(), ref.detach(), rtol=1e-6, atol=1e-6)
    for b in (pb, mb, vb):
        assert torch.all(b[shift + n:] == 7.0) and torch.all(b[:shift] == 7.0)
