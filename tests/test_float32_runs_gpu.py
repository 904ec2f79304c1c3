"""float32 throughout at head dim 64, W <= 64: dK / dV over runs of key tiles
(more tiles than workgroups per (b, h), T ragged so a run ends on a partial
tile), against the float64 oracle at the float32 bound of the other tests."""
import math

import pytest
import torch

from tests._util import make_inputs
from tests.test_window_gpu import check_fp32, hip_run, last_kernel, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,W,normalize,bias,dtau", [
    (1000, 64, "mass", False, False), (1000, 33, "count", True, False), (961, 64, None, False, True),
    (1024, 1, "mass", True, True)])
def test_float32_backward_runs(dev, T, W, normalize, bias, dtau):
    from bozo_amd import _lib as L
    B, H, D = 32, 4, 64
    inp = make_inputs(B, T, H, D, seed=T + W, std=0.5, W=W, dtau_std=0.1 if dtau else None,
                      bias_std=0.5 if bias else None, bias_shape=(B, T, W) if bias else None)
    hip = hip_run(inp, W, math.sqrt(D), dev, normalize=normalize, return_tau=dtau, use_bias=bias, use_dtau=dtau)
    assert last_kernel() == L.KERNEL_SPLIT_F32V
    ref = oracle_run(inp, W, math.sqrt(D), normalize=normalize, use_bias=bias, use_dtau=dtau)
    for name, got, want in zip(("out", "dQ", "dK", "dV"), (hip[0], *hip[2]), (ref[0], *ref[2])):
        check_fp32(got, want, name)
