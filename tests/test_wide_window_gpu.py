"""bf16 local windows wider than one 64-row tile at head dim 64 (the wide band
kernels) against the float64 oracle: windows on and off the 64-key blocks, one
block to the whole sequence, ragged and one-tile sequences, heads that do not
fill the XCDs, every normalisation, K / V as views of one projection.  P and G
enter the second products in bf16 and results are rounded to bf16 from float32
sums, so a result differs from float64 by about 2^-8.5 relative L2 (measured
2.2e-3 to 2.6e-3 here and on the split kernels these calls ran on before); 4e-3
admits that.  With side operands the calls stay on the split kernels."""
import pytest
import torch

from tests._util import f64, make_inputs, rel_l2
from tests.test_window_gpu import hip_run, last_kernel, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normalize", ["mass", "count", None])
@pytest.mark.parametrize("B,T,H,W", [(2, 1, 3, 65), (1, 64, 2, 100), (2, 65, 3, 65), (1, 200, 8, 128), (2, 333, 3, 129),
                                     (1, 777, 4, 256), (1, 500, 2, 300), (1, 192, 8, 1000), (1, 129, 1, 127)])
def test_wide_window(dev, B, T, H, W, normalize):
    from bozo_amd import _lib as L
    inp = make_inputs(B, T, H, 64, seed=T + W, std=0.7, dtype=torch.bfloat16, W=W)
    hip = hip_run(inp, W, 8.0, dev, normalize=normalize)
    assert last_kernel() == L.KERNEL_MFMA
    ref = oracle_run(inp, W, 8.0, normalize=normalize)
    for name, got, want in zip(("out", "dQ", "dK", "dV"), (hip[0], *hip[2]), (ref[0], *ref[2])):
        assert rel_l2(f64(got), want) <= 4e-3, name


@pytest.mark.parametrize("normalize", ["mass", "count", None])
def test_wide_window_matches_split_kernels(dev, normalize):
    """The same call with a zero bias runs on the split kernels: the route does
    not show beyond rounding; K and V as views of one projection."""
    from bozo_amd import _lib as L
    from bozo_amd import causal_tension
    B, T, H, W = 2, 450, 4, 200
    g = torch.Generator().manual_seed(3)
    q = torch.randn(B, T, H, 64, generator=g).to(torch.bfloat16).to(dev).requires_grad_(True)
    kv = torch.randn(B, T, H, 128, generator=g).to(torch.bfloat16).to(dev)
    k, v = (x.detach().requires_grad_(True) for x in kv.split(64, -1))
    do = torch.randn(B, T, H, 64, generator=g).to(torch.bfloat16).to(dev)
    res = []
    for bias, kernel in ((None, L.KERNEL_MFMA), (torch.zeros(B, T, W, device=dev), L.KERNEL_SPLIT_BF16)):
        out = causal_tension(q, k, v, W, 8.0, bias=bias, normalize=normalize)
        assert last_kernel() == kernel
        res.append([out, *torch.autograd.grad(out, [q, k, v], do)])
    for a, b in zip(*res):
        assert rel_l2(f64(a), f64(b)) <= 2.0 ** -8


def test_wide_window_mass_without_normalisation(dev):
    """The C API's tau mass beside a valid-count output (only the split kernels
    write it) is the mass of the tau-mass call."""
    from bozo_amd import _lib as L
    B, T, H, W = 1, 150, 2, 100
    q, k, v = (torch.randn(B, T, H, 64, device=dev).to(torch.bfloat16) for _ in range(3))
    out, got = torch.empty_like(q), []
    for flag, kernel in ((L.NORM_MASS, L.KERNEL_MFMA), (L.NORM_COUNT, L.KERNEL_SPLIT_BF16)):
        mass = torch.full((B, T, H), -1.0, device=dev)
        L.check(L.lib().tension_window_fwd(L.buf(q), L.buf(k), L.buf(v), L.buf(out), None, None, L.buf(mass), B, T, H,
                                           64, W, 8.0, flag, L.stream_handle(q.device)), "fwd")
        assert last_kernel() == kernel
        got.append(mass)
    torch.cuda.synchronize()
    assert float((got[0] - got[1]).abs().max()) <= 1e-5 * W
