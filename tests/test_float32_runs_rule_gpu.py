"""float32 throughout at head dim 64, W <= 64, dK / dV on both sides of the line
between runs of key tiles and one tile per workgroup: (b, h) counts that fill the
workgroups two per CU take, leave a round nearly empty, or need more than one round;
with a bias and a dTau the line lies higher.  First and last (b, h) against the
float64 oracle at the float32 bound of the other tests."""
import math

import pytest
import torch

from tests._util import device_cus, make_inputs
from tests.test_window_gpu import check_fp32, hip_run, last_kernel, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias,dtau", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("per_cu,T", [(0.75, 250), (1.0, 130), (1.25, 130), (2.0, 70), (2.01, 130), (3.0, 70)])
def test_either_side_of_the_line(dev, per_cu, T, bias, dtau):
    from bozo_amd import _lib as L
    B, H, D, W = int(per_cu * device_cus() + 0.5) // 2 + 1, 2, 64, 50
    inp = make_inputs(B, T, H, D, seed=B + T, std=0.5, W=W, dtau_std=0.1 if dtau else None,
                      bias_std=0.5 if bias else None, bias_shape=(B, T, W) if bias else None)
    kw = dict(normalize="mass", use_bias=bias, use_dtau=dtau)
    hip = hip_run(inp, W, math.sqrt(D), dev, return_tau=dtau, **kw)
    assert last_kernel() == L.KERNEL_SPLIT_F32V
    ends = {n: None if t is None else t[[0, -1]] for n, t in inp.items()}
    ref = oracle_run(ends, W, math.sqrt(D), **kw)
    for name, got, want in zip(("out", "dQ", "dK", "dV"), (hip[0], *hip[2]), (ref[0], *ref[2])):
        check_fp32(got[[0, -1]], want, name)
