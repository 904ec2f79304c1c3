"""The native autograd nodes of the eager path against the Python Functions
that torch.jit tracing still takes: the same kernels with the same arguments,
so outputs and gradients are equal bit for bit, whatever the layout of the
inputs, the stream, saved-tensor hooks, or which outputs are used."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

W, SCALE = 24, 8.0


def _qkv(dev, qk=torch.float32, v=torch.bfloat16, D=64, T=70, layout="own", grad=True):
    g = torch.Generator().manual_seed(5)
    B, H = 2, 3
    if layout == "fused":
        q, kv = torch.randn(B, T, H, D, generator=g), torch.randn(B, T, H, 2 * D, generator=g)
        k, vv = kv.to(qk).to(dev).split(D, -1)
        ts = [q.to(qk).to(dev), k, vv]
    elif layout == "features_first":  # no unit innermost stride: copied by the op
        ts = [torch.randn(B, D, T, H, generator=g).to(dt).to(dev).permute(0, 2, 3, 1) for dt in (qk, qk, v)]
    else:
        ts = [torch.randn(B, T, H, D, generator=g).to(dt).to(dev) for dt in (qk, qk, v)]
    return [t.detach().requires_grad_(grad) for t in ts]


def _both(ops, monkeypatch, f):
    got = f()
    with monkeypatch.context() as m:
        m.setattr(ops, "_eager", lambda: False)
        want = f()
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("layout", ["own", "fused", "features_first"])
@pytest.mark.parametrize("qk,v,D,win", [(torch.float32, torch.bfloat16, 64, W), (torch.float32, torch.bfloat16, 32, 90),
                                        (torch.float32, torch.float32, 64, W), (torch.bfloat16, torch.bfloat16, 64, 64),
                                        (torch.float16, torch.float16, 32, W), (torch.float64, torch.float64, 16, W)])
@pytest.mark.parametrize("norm,use", [("mass", "both"), ("count", "out"), (None, "tau")])
def test_window_nodes(dev, monkeypatch, layout, qk, v, D, win, norm, use):
    from bozo_amd import ops
    q, k, vv = _qkv(dev, qk, v, D, layout=layout)
    bias = torch.randn(2, 70, win, device=dev) if use == "both" else None

    def f():
        out, tau = ops.causal_tension(q, k, vv, win, math.sqrt(D), return_tau=True, bias=bias, normalize=norm)
        used = {"both": [out, tau], "out": [out], "tau": [tau]}[use]
        return [out, tau, *torch.autograd.grad(used, [q, k, vv], [torch.ones_like(t) for t in used])]

    if use == "both":
        _both(ops, monkeypatch, f)
        return
    # an unused output's gradient is absent here and zeros there: another
    # kernel variant, equal to rounding
    got = f()
    monkeypatch.setattr(ops, "_eager", lambda: False)
    for a, b in zip(got, f()):
        tol = {torch.float64: 1e-12, torch.float32: 1e-5}.get(a.dtype, 4e-2)
        assert a.dtype == b.dtype and float((a.double() - b.double()).abs().max()) <= tol * max(
            1.0, float(b.double().abs().max()))


@pytest.mark.parametrize("dtype,Wl", [(torch.bfloat16, 64), (torch.bfloat16, None), (torch.float32, 7)])
def test_global_nodes(dev, monkeypatch, dtype, Wl):
    from bozo_amd import ops
    q, k, v = _qkv(dev, dtype, dtype)
    bias = torch.randn(2, 70, 70, device=dev) if Wl else None

    def f():
        res = ops.global_tension(q, k, v, SCALE, bias=bias, W_local=Wl)
        outs = list(res) if Wl else [res]
        return [*outs, *torch.autograd.grad(outs, [q, k, v], [torch.ones_like(t) for t in outs])]

    _both(ops, monkeypatch, f)


@pytest.mark.parametrize("out_dtype", [None, torch.float32])
def test_rope_node(dev, monkeypatch, out_dtype):
    from bozo_amd import ops
    x = torch.randn(2, 9, 3, 64, device=dev, dtype=torch.bfloat16, requires_grad=True)
    ang = torch.rand(16, 32, device=dev)

    def f():
        y = ops.rope(x, ang.cos(), ang.sin(), 3, out_dtype)
        return [y, *torch.autograd.grad(y, x, torch.ones_like(y))]

    _both(ops, monkeypatch, f)


def test_side_stream_hooks_and_checkpoint(dev):
    """A backward on the forward's side stream, saved tensors packed to the
    host and back, and a recomputed forward give the plain call's gradients."""
    from torch.utils.checkpoint import checkpoint

    from bozo_amd import causal_tension
    q, k, v = _qkv(dev)
    f = lambda: causal_tension(q, k, v, W, SCALE, normalize="mass")  # noqa: E731
    want = torch.autograd.grad(f().sum(), [q, k, v])
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        got = torch.autograd.grad(f().sum(), [q, k, v])
    s.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.autograd.graph.save_on_cpu():
        out = f()
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(out.sum(), [q, k, v]), want))
    got = torch.autograd.grad(checkpoint(lambda a, b, c: causal_tension(a, b, c, W, SCALE, normalize="mass"), q, k, v,
                                         use_reentrant=False).sum(), [q, k, v])
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_refused_calls(dev):
    from bozo_amd import causal_tension, decode_step, global_tension
    from bozo_amd._lib import TensionError
    q, k, v = _qkv(dev, grad=False)
    with pytest.raises(TypeError):
        causal_tension(q.int(), k.int(), v.int(), W, SCALE)
    with pytest.raises(ValueError):
        causal_tension(q, k, v, W, SCALE, bias=torch.zeros(2, 70, W + 1, device=dev))
    with pytest.raises(ValueError):
        global_tension(q, k, v, SCALE, bias=torch.zeros(2, 70, 71, device=dev))
    with pytest.raises(TensionError):
        causal_tension(q, k, v, W, float("nan"))
    with pytest.raises(RuntimeError):  # no functorch rule, as for a Function without setup_context
        torch.vmap(lambda a: causal_tension(a, k, v, W, SCALE))(torch.stack([q, q]))
    row, cache, pos = q[:, 0], torch.zeros(2, 3, 8, 64, device=dev), torch.zeros(2, dtype=torch.int32, device=dev)
    with pytest.raises(TypeError):
        decode_step(row.int(), row.int(), row.int(), cache.int(), cache.int(), pos, None, SCALE)
    with pytest.raises(ValueError):
        decode_step(row, row, row, cache, cache, pos, None, SCALE, normalize="other")
    with pytest.raises(TensionError):
        decode_step(row, row, row, cache, cache, pos, pos, SCALE)


def test_traced_call_replays(dev):
    """torch.jit.trace records the call, not its first result."""
    from bozo_amd import causal_tension
    q, k, v = _qkv(dev, grad=False)
    f = torch.jit.trace(lambda a, b, c: causal_tension(a, b, c, W, SCALE, normalize="mass"), (q, k, v),
                        check_trace=False)
    q2 = torch.randn_like(q)
    assert torch.equal(f(q2, k, v), causal_tension(q2, k, v, W, SCALE, normalize="mass"))
