"""bf16 windows wider than 64 at head dim 64 without side operands: which kernels
each phase takes -- wide band kernels or split kernels, by the grid's workgroups
per CU and the window -- and that every mix of the two gives the float64 oracle's
results (they hand the coefficients on in one workspace).  Bound as for the wide
kernels: relative L2 2^-8.5 of bf16 weights and results, 4e-3 admits it."""
import pytest
import torch

from tests._util import device_cus, f64, make_inputs, rel_l2
from tests.test_window_gpu import oracle_run

pytestmark = pytest.mark.gpu

# B, H, T, W, phases (forward, dQ, dK / dV) on the wide kernels; tiles per CU
CASES = [
    (1, 4, 300, 65, (1, 1, 1)),  # under one
    (8, 8, 320, 95, (0, 0, 0)), (8, 8, 320, 96, (1, 1, 0)), (8, 8, 320, 128, (1, 1, 1)), (16, 16, 95, 4096, (0, 0, 0)),  # two
    (6, 16, 400, 95, (0, 0, 0)), (6, 16, 400, 96, (1, 0, 0)), (6, 16, 400, 383, (1, 1, 0)), (6, 16, 400, 384, (1, 1, 1)),  # three
    (9, 16, 300, 4096, (1, 0, 0)),
    (8, 16, 400, 127, (0, 0, 0)), (8, 16, 400, 128, (1, 0, 1)), (8, 16, 400, 256, (1, 1, 1)),  # four
    (10, 16, 500, 255, (1, 0, 0)), (10, 16, 500, 256, (1, 1, 1)),  # five
    (12, 16, 600, 127, (0, 0, 0)), (12, 16, 600, 128, (1, 0, 1)), (12, 16, 600, 320, (1, 1, 1)),  # eight
    (60, 16, 150, 4096, (1, 0, 0)), (48, 16, 330, 320, (1, 0, 0)),  # twelve, eighteen
]


@pytest.mark.parametrize("norm", ["mass", "count"])
@pytest.mark.parametrize("B,H,T,W,wide", CASES)
def test_route_and_mixed_phases(dev, B, H, T, W, wide, norm):
    from bozo_amd import _lib as L
    if device_cus() != 256:
        pytest.skip("the cases are laid out for 256 CUs")
    inp = make_inputs(B, T, H, 64, seed=B + W, std=0.7, dtype=torch.bfloat16)
    q, k, v, do = (inp[n].to(dev) for n in ("Q", "K", "V", "dO"))
    out, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
    flag = L.NORM_MASS if norm == "mass" else L.NORM_COUNT
    lib, st = L.lib(), L.stream_handle(q.device)
    ws = torch.empty(max(1, lib.tension_window_bwd_workspace(B, T, H, L.F32, flag)), dtype=torch.uint8, device=dev)
    dims, kernels, b = (B, T, H, 64, W, 8.0, flag, st), [], L.buf

    def phase(status):
        L.check(status, "phase")
        kernels.append(int(lib.tension_last_kernel()))

    phase(lib.tension_window_fwd(b(q), b(k), b(v), b(out), None, None, None, *dims))
    phase(lib.tension_window_bwd_dq(b(q), b(k), b(v), b(do), None, None, b(dq), ws.data_ptr(), *dims))
    phase(lib.tension_window_bwd_dkv(b(q), b(k), b(v), b(do), None, None, b(dk), b(dv), ws.data_ptr(), *dims))
    assert kernels == [L.KERNEL_MFMA if w else L.KERNEL_SPLIT_BF16 for w in wide]

    def pick(t):  # the last head of the first and the last sequence
        return t[[0, B - 1] if B > 1 else [0]][:, :, H - 1:]

    want = oracle_run({n: pick(inp[n]) for n in ("Q", "K", "V", "dO")}, W, 8.0, normalize=norm)
    for name, got, ref in zip(("out", "dQ", "dK", "dV"), (out, dq, dk, dv), (want[0], *want[2])):
        assert rel_l2(f64(pick(got)), ref) <= 4e-3, name


def test_long_sequence(dev):
    """All three wide kernels over 625 tiles, in segments."""
    from bozo_amd import _lib as L
    from tests.test_long_seq_gpu import test_window_long_sequence_segments as segments
    segments(dev, torch.bfloat16, 40000, 1, 300, "mass")
    assert int(L.lib().tension_last_kernel()) == L.KERNEL_MFMA
