"""tau_local / dtau_local of the bf16 global kernels over the blocks that hold
their columns: one key, a block's edge on either side, several blocks, every key;
whole and ragged last tiles.  dtau_local at the scale of dP, so a value at a wrong
pair shows in dQ and dK."""
import pytest
import torch

from tests._util import make_inputs
from tests.test_global_gpu import check, hip_run, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("T,wl", [(1, 1), (64, 64), (65, 1), (128, 63), (128, 65), (190, 62), (190, 64), (191, 128),
                                  (257, 257), (320, 200)])
def test_tau_blocks(dev, T, wl, bias):
    inp = make_inputs(2, T, 3, 64, seed=T + wl, std=0.5, dtype=torch.bfloat16, W=wl, dtau_std=1.0,
                      bias_std=0.5 if bias else None, bias_shape=(2, T, T) if bias else None)
    kw = dict(W_local=wl, use_bias=bias, use_dtl=True)
    check(hip_run(inp, 8.0, dev, **kw), oracle_run(inp, 8.0, **kw), torch.bfloat16, True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.float64])
def test_dtau_types(dev, dtype):
    """A dtau_local of another type with the same values gives the same bits."""
    from bozo_amd import _lib
    B, T, H, wl = 2, 150, 3, 70
    g = torch.Generator().manual_seed(5)
    Q, K, V, dO = (torch.randn(B, T, H, 64, generator=g).to(torch.bfloat16).to(dev) for _ in range(4))
    dtl = (torch.randint(-64, 65, (B, T, H, wl), generator=g) / 64).to(dev)
    host = _lib.host()
    out, _, mass = host.global_fwd(Q, K, V, None, 8.0, 0)
    want = host.global_bwd(Q, K, V, dO, dtl.to(torch.bfloat16), None, out, mass, wl, 8.0)
    got = host.global_bwd(Q, K, V, dO, dtl.to(dtype), None, out, mass, wl, 8.0)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
