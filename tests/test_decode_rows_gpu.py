"""Decode steps outside the head-dim-64 fast kernel, against the float64
oracle: the row kernel (aligned rows of 32, 64 and 128 elements) around the
edges of its trips -- 256, 128 and 64 rows at head dims 32, 64 and 128 with 4
waves, four times that with 16 (a long cache on a small grid) -- and the general one (other head dims, mixed dtypes, unaligned rows).  Dead
slots hold NaN: they are nobody's rows and must not be read into a result.

Tolerances: float32 sums of W products of the float32 inputs differ from
float64 by at most about W 2^-24 of the largest term, normalised outputs by
a few 2^-24 of |out| <= 4 (1e-5, the bound of the other float32 tests); 16-bit
outputs by half a unit of their own type (relative L2 2^-9 / 2^-12, tau
likewise).
"""
import math

import numpy as np
import pytest
import torch

from oracle import tension_oracle as O
from tests._util import f64, max_abs, rel_l2

pytestmark = pytest.mark.gpu

_F32, _BF16, _F16, _F64 = torch.float32, torch.bfloat16, torch.float16, torch.float64

# q / K dtype, V dtype, D, W, positions, self key, tau, storage offset of every tensor's rows, heads
CASES = [
    (_F32, _F32, 64, 1024, (0, 1, 511, 512, 513, 1023), True, False, 0),
    (_F32, _F32, 64, 300, (127, 128, 129, 256), True, False, 0, 130),      # 4 waves, several trips
    (_BF16, _BF16, 32, 600, (255, 256, 257, 700), False, True, 0, 130),
    (_F32, _BF16, 128, 130, (63, 64, 65, 128, 131), False, True, 0, 110),
    (_F32, _F32, 64, 600, (0, 3, 511, 600, 601, 1500), False, True, 0),
    (_BF16, _BF16, 64, 1500, (0, 1, 256, 700, 1499, 2900), False, True, 0),
    (_BF16, _BF16, 64, 2048, (1, 1030, 2047), True, False, 0),
    (_F32, _BF16, 64, 1100, (0, 5, 512, 1099, 1101), False, True, 0),
    (_F32, _BF16, 64, 64, (0, 31, 63), True, False, 0),
    (_F16, _F16, 32, 520, (0, 2, 511, 513, 700), False, True, 0),
    (_F32, _F32, 32, 8, (0, 3, 8, 21), False, True, 0),
    (_BF16, _BF16, 32, 513, (0, 512), True, False, 0),
    (_F32, _F32, 128, 129, (0, 127, 128, 129, 400), False, True, 0),
    (_F16, _F16, 128, 300, (0, 1, 299), True, False, 0),
    (_F32, _F32, 20, 70, (0, 4, 63, 64, 65, 141), False, True, 0),       # no vector head dim
    (_F32, _F32, 64, 70, (0, 5, 69), True, False, 1),                     # rows off their 16 bytes
    (_F32, _F16, 256, 33, (0, 17, 80), False, True, 0),                   # mixed dtypes, the largest D
    (_F64, _F64, 1, 5, (0, 2, 9), False, True, 0),
    (_F64, _F64, 64, 40, (0, 15, 39), True, False, 0),
]


@pytest.mark.parametrize("norm", ["mass", "count", "raw"])
@pytest.mark.parametrize("case", CASES, ids=[f"{str(c[0])[6:]}-{str(c[1])[6:]}-D{c[2]}W{c[3]}"
                                             f"{'-self' if c[5] else ''}{'-off' if c[7] else ''}-H{(*c, 3)[8]}" for c in CASES])
def test_decode_rows(dev, case, norm):
    from bozo_amd import decode_step
    qd, vd, D, W, where, self_key, want_tau, off, H = (*case, 3)[:9]
    N = len(where)
    g = torch.Generator().manual_seed(41 + W + D)
    print(f"[decode rows {case} {norm}]", flush=True)

    def rows(*shape, dt):
        return torch.randn(*shape, generator=g, dtype=torch.float64).mul(0.5).to(dt)

    def on_gpu(x):
        if not off:
            return x.to(dev)
        buf = torch.empty(*x.shape[:-1], x.shape[-1] + off, dtype=x.dtype, device=dev)[..., off:]
        return buf.copy_(x)

    q, kn, vn = rows(N, H, D, dt=qd), rows(N, H, D, dt=qd), rows(N, H, D, dt=vd)
    kc, vc = rows(N, H, W, D, dt=qd), rows(N, H, W, D, dt=vd)
    pos = np.asarray(where, np.int32)
    ref, rt = O.decode_step(f64(q), f64(kc), f64(vc), pos, W, math.sqrt(D), norm if norm != "raw" else False,
                            (f64(kn), f64(vn)) if self_key else None)
    for n, p in enumerate(where):
        kc[n, :, min(p, W):] = float("nan")
        vc[n, :, min(p, W):] = float("nan")
    gk, gv = on_gpu(kc), on_gpu(vc)
    pin = torch.from_numpy(pos).to(dev)
    pout = torch.empty_like(pin)
    tau = torch.empty(N, H, W, dtype=qd, device=dev) if want_tau else None
    out = decode_step(on_gpu(q), on_gpu(kn), on_gpu(vn), gk, gv, pin, pout, math.sqrt(D), norm, tau, self_key)
    torch.cuda.synchronize()
    if qd in (_F32, _F64):
        lim = 1e-9 if qd == _F64 else 1e-5 * max(1.0, float(np.abs(ref).max()))
        assert max_abs(f64(out), ref) <= lim
    else:
        assert rel_l2(f64(out), ref) <= (2.0 ** -9 if qd == _BF16 else 2.0 ** -12)
    if want_tau:
        lim = {_F64: 1e-9, _F32: 1e-6, _BF16: 2.0 ** -9 + 1e-6, _F16: 2.0 ** -12 + 1e-6}[qd]
        assert max_abs(f64(tau), rt) <= lim
    for n, p in enumerate(where):  # only slot pos % W changed, to the new token's rows
        kc[n, :, p % W], vc[n, :, p % W] = kn[n], vn[n]
    assert torch.equal(gk.cpu().nan_to_num(9.0), kc.nan_to_num(9.0))
    assert torch.equal(gv.cpu().nan_to_num(9.0), vc.nan_to_num(9.0))
    assert pout.cpu().tolist() == [p + 1 for p in where]
