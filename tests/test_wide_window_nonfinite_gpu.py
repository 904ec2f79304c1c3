"""Non-finite rows in the wide band kernels (bf16, head dim 64, W > 64, no side
operands).  A masked pair is weight 0 times its row, so a NaN or infinity may
reach a result row without a pair with it, but only within a product: 16 result
rows against 32 summed rows, left out where the band does not touch them.  Every
result row outside those groups is the finite call's bit for bit, and every row
with a pair is not."""
import math

import pytest
import torch

from tests._util import make_inputs
from tests.test_window_gpu import last_kernel

pytestmark = pytest.mark.gpu

T, W = 400, 300


def _band(q, k):
    return 0 <= k < q < T and k >= q - W


def _reach(row, row_is_query):
    """Result rows whose 16-row group has a pair with the 32-row group of `row`."""
    g32 = range(row // 32 * 32, row // 32 * 32 + 32)
    out = set()
    for a in range(0, T, 16):
        pairs = ((r, x) if row_is_query else (x, r) for x in range(a, a + 16) for r in g32)
        if any(_band(q, k) for q, k in pairs):
            out |= set(range(a, min(a + 16, T)))
    return out


@pytest.mark.parametrize("normalize", ["count", "mass", None])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("operand", ["Q", "K", "V", "dO"])
def test_reach_of_a_nonfinite_row(dev, operand, value, normalize):
    from bozo_amd import _lib as L
    from bozo_amd import causal_tension

    def run(row):
        inp = make_inputs(1, T, 2, 64, seed=7, std=0.7, dtype=torch.bfloat16)
        if row is not None:
            inp[operand][:, row, 0, 5] = value  # one element: head 0 only
        q, k, v = (inp[n].to(dev).requires_grad_() for n in "QKV")
        out = causal_tension(q, k, v, W, math.sqrt(64), normalize=normalize)
        assert last_kernel() == L.KERNEL_MFMA
        return [out, *torch.autograd.grad(out, [q, k, v], inp["dO"].to(dev))]

    clean = run(None)
    for row in (0, 17, 40, 63, 130, 350, 399):
        query = operand in ("Q", "dO")
        with_pair = {x for x in range(T) if (_band(row, x) if query else _band(x, row))}
        by_group = _reach(row, query)
        if normalize == "mass" and not query:
            # the row's queries carry it in their coefficients to all their keys
            by_group |= {k for q in with_pair for k in range(max(0, q - W), q)}
        for name, a, b in zip(("out", "dQ", "dK", "dV"), run(row), clean):
            assert torch.equal(a[:, :, 1], b[:, :, 1]), (name, row)  # the other head
            same = (a[0, :, 0] == b[0, :, 0]).all(-1).cpu()
            changed = {int(x) for x in torch.nonzero(~same)[:, 0]}
            assert changed <= by_group | {row}, (name, row, sorted(changed - by_group))
        # dO enters dV and V enters out, K enters dQ and Q enters dK: their rows with a pair are not finite
        hit = {"Q": 2, "K": 1, "V": 0, "dO": 3}[operand]
        got = run(row)[hit][0, :, 0]
        bad = {int(x) for x in torch.nonzero(~torch.isfinite(got).all(-1))[:, 0]}
        assert with_pair <= bad, (row, sorted(with_pair - bad))
