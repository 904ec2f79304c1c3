"""The split forward with one key group per workgroup (the grids of real batches)
and with two (small grids), each against the float64 oracle and each seen to run:
a batch past the line as one call, its first and last sequence alone.

Bounds: float32 rows, the float32 bound of the other tests at |out| <= 4 and in
proportion above (raw sums); bf16 and float16, the rounding of a result and, in
bf16, of the weights that enter the second product (relative L2 2^-8.5 and 2^-12:
4e-3 and 2^-11 admit them)."""
import numpy as np
import pytest
import torch

from tests._util import device_cus, f64, make_inputs, max_abs, rel_l2
from tests.test_global_gpu import oracle_run as global_oracle
from tests.test_window_gpu import oracle_run as window_oracle

pytestmark = pytest.mark.gpu

_DT = {"bf16": (torch.bfloat16, torch.bfloat16), "autocast": (torch.float32, torch.bfloat16),
       "f32": (torch.float32, torch.float32), "f16": (torch.float16, torch.float16)}


def _close(got, want, dtype, what):
    if dtype == torch.float32:
        assert max_abs(f64(got), want) <= 1e-5 * max(1.0, float(np.abs(want).max()) / 4), what
    else:
        assert rel_l2(f64(got), want) <= (4e-3 if dtype == torch.bfloat16 else 2.0 ** -11), what


@pytest.mark.parametrize("normalize", ["count", None, "mass"])
@pytest.mark.parametrize("flow,D,T,W,tau", [
    ("autocast", 64, 300, 256, True), ("autocast", 32, 130, 100, False), ("f32", 64, 257, 65, True),
    ("f32", 32, 200, 128, False), ("f16", 64, 200, 129, True), ("f16", 32, 129, 400, False),
    ("bf16", 32, 300, 200, True), ("bf16", 64, 190, 70, True)])
def test_window_groups(dev, flow, D, T, W, tau, normalize):
    from bozo_amd import _lib as L
    from bozo_amd import causal_tension
    qk, v = _DT[flow]
    H = 8
    B = 2 * device_cus() // (H * ((T + 63) // 64)) + 1
    inp = make_inputs(B, T, H, D, seed=T + W, std=0.6)
    t = {n: inp[n].to(v if n == "V" else qk) for n in ("Q", "K", "V", "dO")}
    g = {n: x.to(dev) for n, x in t.items()}
    for groups, picks in ((1, [slice(None)]), (2, [slice(0, 1), slice(B - 1, B)])):
        for s in picks:
            res = causal_tension(g["Q"][s], g["K"][s], g["V"][s], W, D ** 0.5, return_tau=tau, normalize=normalize)
            assert int(L.lib().tension_last_key_groups()) == groups
            ends = [0, B - 1] if groups == 1 else [s.start]
            ref = window_oracle({n: x[ends] for n, x in t.items()}, W, D ** 0.5, normalize=normalize)
            out = res[0] if tau else res
            _close(out[[0, -1]] if groups == 1 else out, ref[0], qk, "out")
            if tau:
                _close(res[1][[0, -1]] if groups == 1 else res[1], ref[1], qk, "tau")


@pytest.mark.parametrize("flow,D,T", [("f32", 64, 200), ("f16", 32, 129), ("bf16", 32, 190), ("autocast", 64, 130)])
def test_global_groups(dev, flow, D, T):
    from bozo_amd import _lib as L
    from bozo_amd import global_tension
    qk, v = _DT[flow]
    H = 8
    B = 2 * device_cus() // (H * ((T + 63) // 64)) + 1
    inp = make_inputs(B, T, H, D, seed=T, std=0.6)
    t = {n: inp[n].to(v if n == "V" else qk) for n in ("Q", "K", "V", "dO")}
    g = {n: x.to(dev) for n, x in t.items()}
    for groups, s, ends in ((1, slice(None), [0, B - 1]), (2, slice(B - 1, B), [B - 1])):
        out, tl = global_tension(g["Q"][s], g["K"][s], g["V"][s], D ** 0.5, W_local=50)
        assert int(L.lib().tension_last_key_groups()) == groups
        ref = global_oracle({n: x[ends] for n, x in t.items()}, D ** 0.5, W_local=50)
        pick = [0, -1] if groups == 1 else [0]
        _close(out[pick], ref[0], qk, "out")
        _close(tl[pick], ref[1], qk, "tau_local")
