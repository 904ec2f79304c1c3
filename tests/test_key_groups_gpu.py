"""The split kernels' forward with one and with two key groups per workgroup
(small grids take two): a batch whose tiles pass the line is computed as one
call and sequence by sequence, and the two agree to the rounding of one more
float32 addition -- |out|, tau <= 4 and a few sums of up to W terms: 1e-5
(float32 rows), one unit of the type otherwise.  tau columns, empty slots and
bias land alike."""
import pytest
import torch

from tests._util import device_cus

pytestmark = pytest.mark.gpu

_DT = {"bf16": (torch.bfloat16, torch.bfloat16), "autocast": (torch.float32, torch.bfloat16),
       "f32": (torch.float32, torch.float32), "f16": (torch.float16, torch.float16)}


@pytest.mark.parametrize("flow,D,T,W,tau,bias", [
    ("autocast", 64, 300, 256, True, True), ("autocast", 64, 65, 100, False, False), ("f32", 64, 257, 65, True, False),
    ("f32", 32, 130, 128, False, True), ("f16", 64, 200, 129, True, True), ("bf16", 64, 300, 200, True, False),
    ("bf16", 32, 64, 66, False, True), ("autocast", 32, 500, 400, True, False),
    ("f32", 64, 300, None, True, True), ("f16", 32, 129, None, False, False), ("bf16", 32, 190, None, True, False)])
def test_key_groups_agree(dev, flow, D, T, W, tau, bias):
    from bozo_amd import causal_tension, global_tension
    qk, v = _DT[flow]
    H, tiles = 16, (T + 63) // 64
    B = 2 * device_cus() // (H * tiles) + 1  # past the line as one batch, below it alone
    assert B > 1
    g = torch.Generator().manual_seed(T)
    Q, K, V = (torch.randn(B, T, H, D, generator=g).to(dt).to(dev) for dt in (qk, qk, v))
    Bias = torch.randn(B, T, W or T, generator=g).to(dev) if bias else None

    def call(b):
        s = slice(None) if b is None else slice(b, b + 1)
        args = Q[s], K[s], V[s]
        bb = None if Bias is None else Bias[s]
        if W is None:
            res = global_tension(*args, D ** 0.5, bias=bb, W_local=min(50, T) if tau else None)
        else:
            res = causal_tension(*args, W, D ** 0.5, return_tau=tau, bias=bb, normalize="mass")
        return res if tau else (res,)

    whole = call(None)
    for b in (0, B - 1):
        for x, y in zip(whole, call(b)):
            x = x[b:b + 1]
            assert x.shape == y.shape and bool(torch.equal(x == 0, y == 0))
            lim = 1e-5 if qk == torch.float32 else 2.0 ** -7 if qk == torch.bfloat16 else 2.0 ** -9
            assert float((x.double() - y.double()).abs().max()) <= lim
