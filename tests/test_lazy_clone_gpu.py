"""A decode step on tensors that share their memory lazily (torch._lazy_clone:
one storage until somebody asks for a mutable pointer): what the step writes --
the caches, tau, pos_out -- lands in the tensor it was given and in no other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step_on", ["clone", "original"])
@pytest.mark.parametrize("dtype,D,W", [(torch.bfloat16, 64, 16), (torch.float32, 32, 8)])
def test_step_on_shared_caches(dev, step_on, dtype, D, W):
    from bozo_amd import decode_step
    N, H = 2, 3
    g = torch.Generator().manual_seed(9)
    q, kn, vn = (torch.randn(N, H, D, generator=g).to(dtype).to(dev) for _ in range(3))
    k, v = (torch.randn(N, H, W, D, generator=g).to(dtype).to(dev) for _ in range(2))
    tau = torch.full((N, H, W), -1.0, dtype=dtype, device=dev)
    pos, pout = (torch.full((N,), p, dtype=torch.int32, device=dev) for p in (5, -7))

    want = [t.clone() for t in (k, v, tau, pout)]
    out = decode_step(q, kn, vn, want[0], want[1], pos, want[3], D ** 0.5, tau=want[2])

    first = [k, v, tau, pout]
    before = [t.cpu() for t in first]
    second = [torch._lazy_clone(t) for t in first]
    used, other = (second, first) if step_on == "clone" else (first, second)
    got = decode_step(q, kn, vn, used[0], used[1], pos, used[3], D ** 0.5, tau=used[2])
    torch.cuda.synchronize()
    assert torch.equal(got, out)
    for u, w, o, b in zip(used, want, other, before):
        assert torch.equal(u, w) and not torch.equal(u.cpu(), b)
        assert torch.equal(o.cpu(), b)
