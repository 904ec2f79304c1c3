"""The work a user of bozo_amd gives it, as cases that can be timed and checked.

A case is one of four kinds:

* ``window``  one local tension layer's op: ``causal_tension`` forward, and
  its backward through autograd where ``grad`` is set;
* ``global``  the full-causal block: ``global_tension``, likewise;
* ``decode``  one streaming step over ring K/V caches: ``decode_step``;
* ``layer``   a whole ``MultiHeadCausalTensionLayer`` (projections, RoPE, the
  op, output projection, residual, norm) in training.

``flow`` names the element types: ``bf16`` and ``f16`` throughout;
``autocast`` is the model's own flow (RoPE promotes Q / K to float32, V stays
bf16, so out / dOut / dQ / dK and tau are float32); ``f32`` the model run
without autocast.

Every function takes a case of plain values; inputs come from the seed alone.
"""
from __future__ import annotations

import math

import torch

import bozo_amd
from bozo_amd.model import MultiHeadCausalTensionLayer, TensionConfig

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _qk_dtype(flow):
    return torch.float32 if flow == "autocast" else _DT[flow]


def _v_dtype(flow):
    return torch.bfloat16 if flow == "autocast" else _DT[flow]


def listed():
    return [
        # The smallest training call: the reference's default head dim (32) and
        # BASELINE config 1's shape, float32.  Launches and host work are all of it.
        dict(name="window_small_f32", kind="window", flow="f32", B=4, H=4, T=256, D=32, W=32, norm="mass", tau=False,
             bias=False, kv="own", grad=True),
        # The 117M model's local layer (BASELINE config 2's shape) in bf16 with a
        # batch of 32 sequences: the ordinary training call of the fast_rope model.
        dict(name="window_117m_bf16", kind="window", flow="bf16", B=32, H=12, T=1024, D=64, W=64, norm="mass",
             tau=False, bias=False, kv="own", grad=True),
        # The same layer in the model's default training step: autocast dtypes, tau
        # returned for the aux losses and its gradient coming back.
        dict(name="window_117m_autocast_tau", kind="window", flow="autocast", B=8, H=12, T=1024, D=64, W=64,
             norm="mass", tau=True, bias=False, kv="own", grad=True),
        # The 350M preset's local layer (H16, W256), autocast dtypes.
        dict(name="window_350m_autocast", kind="window", flow="autocast", B=8, H=16, T=1024, D=64, W=256, norm="mass",
             tau=False, bias=False, kv="own", grad=True),
        # The same layer in bf16 on the valid-count path (the 350m preset's --triton
        # training without aux losses).
        dict(name="window_350m_bf16", kind="window", flow="bf16", B=8, H=16, T=1024, D=64, W=256, norm="count",
             tau=False, bias=False, kv="own", grad=True),
        # float32 training without autocast, a ragged sequence length, K and V as
        # views of the fused projection the model without RoPE has.
        dict(name="window_f32_ragged", kind="window", flow="f32", B=8, H=12, T=1000, D=64, W=64, norm="mass",
             tau=False, bias=False, kv="fused", grad=True),
        # Prefill of one prompt of odd length with the graph bias and tau exported,
        # as the streaming exporter runs it: one forward at batch 1.
        dict(name="window_prefill_bias", kind="window", flow="autocast", B=1, H=16, T=777, D=64, W=256, norm="mass",
             tau=True, bias=True, kv="own", grad=False),
        # the global block over 2048 tokens.
        dict(name="global_2048_bf16", kind="global", flow="bf16", B=4, H=12, T=2048, D=64, Wl=0, bias=False,
             grad=True),
        # The 117M model's global layer in its default training step: tau_local out,
        # its gradient back.
        dict(name="global_117m_tau", kind="global", flow="bf16", B=8, H=12, T=1024, D=64, Wl=64, bias=False,
             grad=True),
        # one decode step of 64 sequences at the 350M width.
        dict(name="decode_350m_bf16", kind="decode", flow="bf16", N=64, H=16, D=64, W=256, pos=1000, self_key=False,
             norm="mass", tau=False),
        # Cached generation of a float32 117M model (no autocast): the global layers'
        # step over every earlier token, the new token a key too.
        dict(name="decode_global_f32", kind="decode", flow="f32", N=16, H=12, D=64, W=1024, pos=700, self_key=True,
             norm="mass", tau=False),
        # A whole local layer of the 117M model in the default training step: GEMMs,
        # RoPE, the op with tau, norm, and every gradient.
        dict(name="layer_117m_autocast", kind="layer", flow="autocast", B=8, H=12, T=1024, D=64, W=64),
    ]


# ------------------------------------------------------------------ draws

# relative cost of a (query, key) pair of one flow, about the matrix products it takes
_PAIR_COST = {"bf16": 1.0, "f16": 4.0, "autocast": 5.0, "f32": 6.0}


def _pairs(case):
    """Valid (query, key) pairs."""
    B, H, T = case["B"], case["H"], case["T"]
    if case["kind"] == "global":
        return B * H * T * (T + 1) // 2
    W = case["W"]
    n = min(W, T)
    return B * H * (n * (n - 1) // 2 + (T - n) * W)


def _cost(case):
    """A rough cost of one pass: the rows it reads and the pairs it visits."""
    if case["kind"] == "decode":
        return case["N"] * case["H"] * case["W"] * case["D"] * (2.0 if case["flow"] == "f32" else 1.0)
    rows = case["B"] * case["H"] * case["T"]
    return _PAIR_COST[case["flow"]] * (_pairs(case) + 64 * rows) * case["D"] * (2.0 if case["grad"] else 0.7)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    limit = max(_cost(c) for c in listed() if c["kind"] == "window")
    while True:
        kind = rng.choices(("window", "global", "decode"), (0.6, 0.2, 0.2))[0]
        if kind == "decode":
            flow = rng.choice(("bf16", "autocast", "f32", "f16"))
            self_key = flow != "autocast" and rng.random() < 0.4
            W = rng.choice((256, 512, 1024, 2048)) if self_key else rng.choice((8, 32, 64, 100, 256, 512, 1000))
            pos = _log_int(rng, 1, W - 1) if self_key else _log_int(rng, 1, 4 * W)
            case = dict(kind=kind, flow=flow, N=_log_int(rng, 1, 256), H=rng.choice((4, 12, 16)),
                        D=rng.choice((32, 64, 64)), W=W, pos=pos, self_key=self_key,
                        norm=rng.choice(("mass", "count", "raw")), tau=not self_key and rng.random() < 0.3)
        elif kind == "global":
            T = _log_int(rng, 64, 4096)
            case = dict(kind=kind, flow=rng.choice(("bf16", "bf16", "f32", "f16")), B=_log_int(rng, 1, 16),
                        H=rng.choice((4, 12, 16)), T=T, D=rng.choice((32, 64, 64)),
                        Wl=rng.choice((0, 0, min(64, T))), bias=rng.random() < 0.2, grad=rng.random() < 0.7)
        else:
            case = dict(kind=kind, flow=rng.choice(("bf16", "autocast", "f32", "f16")), B=_log_int(rng, 1, 32),
                        H=rng.choice((1, 4, 12, 16)), T=_log_int(rng, 16, 8192), D=rng.choice((32, 64, 64)),
                        W=rng.choice((8, 32, 64, 64, 100, 128, 256, 256, 400)),
                        norm=rng.choice(("mass", "mass", "count", "raw")), tau=rng.random() < 0.35,
                        bias=rng.random() < 0.2, kv=rng.choice(("own", "fused")), grad=rng.random() < 0.75)
        if _cost(case) <= 0.8 * limit:
            return case


# ------------------------------------------------------------------ inputs

def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _edge_bias(g, *shape):
    """A graph bias: most pairs none, some of them a weight."""
    w = torch.rand(*shape, generator=g, device="cuda")
    on = torch.rand(*shape, generator=g, device="cuda") < 0.05
    return torch.where(on, w, torch.zeros_like(w))


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, flow = case["kind"], case["flow"]
    s = {"case": case}
    if kind == "layer":
        B, T, dim = case["B"], case["T"], case["H"] * case["D"]
        s["x"] = _randn(g, B, T, dim)
        s["weights"] = {n: _randn(g, dim, dim, scale=0.02) for n in ("wq", "wk", "wv", "wo")}
        s["norm_scale"] = 1.0 + _randn(g, dim, scale=0.05)
        s["dout"] = _randn(g, B, T, dim, scale=0.1)
        s["dtau"] = _randn(g, B, T, case["H"], case["W"], scale=0.01)
        return s
    dq, dv, H, D = _qk_dtype(flow), _v_dtype(flow), case["H"], case["D"]
    if kind == "decode":
        N, W = case["N"], case["W"]
        for n, dt in (("q", dq), ("k_new", dq), ("v_new", dv)):
            s[n] = _randn(g, N, H, D, dtype=dt)
        s["k_cache"] = _randn(g, N, H, W, D, dtype=dq)
        s["v_cache"] = _randn(g, N, H, W, D, dtype=dv)
        return s
    B, T = case["B"], case["T"]
    s["Q"] = _randn(g, B, T, H, D, dtype=dq)
    if kind == "window" and case["kv"] == "fused" and dq == dv:
        s["K"], s["V"] = _randn(g, B, T, H, 2 * D, dtype=dq).split(D, dim=-1)
    else:
        s["K"], s["V"] = _randn(g, B, T, H, D, dtype=dq), _randn(g, B, T, H, D, dtype=dv)
    s["dOut"] = _randn(g, B, T, H, D, dtype=dq)
    width = case["W"] if kind == "window" else case["Wl"]
    has_tau = case["tau"] if kind == "window" else case["Wl"] > 0
    s["dTau"] = _randn(g, B, T, H, width, dtype=dq, scale=0.1) if has_tau else None
    s["bias"] = _edge_bias(g, B, T, width if kind == "window" else T) if case["bias"] else None
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "layer":
        cfg = TensionConfig(dim=case["H"] * case["D"], num_heads=case["H"], window=case["W"], max_seq_len=case["T"],
                            dropout=0.0, use_rope=True)
        layer = MultiHeadCausalTensionLayer(cfg).cuda()
        with torch.no_grad():
            for n, w in s["weights"].items():
                getattr(layer, n).weight.copy_(w)
            layer.norm.scale.copy_(s["norm_scale"])
        s["layer"] = layer
        s["x"].requires_grad_(True)
        s["wrt"] = [s["x"]] + [getattr(layer, n).weight for n in ("wq", "wk", "wv", "wo")] + [layer.norm.scale]
    elif case["kind"] == "decode":
        s["pos_in"] = torch.full((case["N"],), case["pos"], dtype=torch.int32, device="cuda")
        s["pos_out"] = torch.zeros(case["N"], dtype=torch.int32, device="cuda")
        if case["tau"]:
            s["tau"] = torch.zeros(case["N"], case["H"], case["W"], dtype=s["q"].dtype, device="cuda")
    elif case["grad"]:
        for n in ("Q", "K", "V"):
            s[n].requires_grad_(True)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    case = s["case"]
    if case["kind"] == "layer":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out, tau = s["layer"](s["x"], return_tensions=True)
        grads = torch.autograd.grad([out, tau], s["wrt"], [s["dout"].to(out.dtype), s["dtau"].to(tau.dtype)])
        return {"out": out, "tau": tau, "grads": list(grads)}
    scale = math.sqrt(case["D"])
    if case["kind"] == "decode":
        tau = s.get("tau")
        out = bozo_amd.decode_step(s["q"], s["k_new"], s["v_new"], s["k_cache"], s["v_cache"], s["pos_in"],
                                   s["pos_out"], scale, normalize=case["norm"], tau=tau,
                                   include_self=case["self_key"])
        return {"out": out, "tau": tau, "k_cache": s["k_cache"], "v_cache": s["v_cache"], "pos": s["pos_out"]}
    tau = None
    with torch.set_grad_enabled(case["grad"]):
        if case["kind"] == "global":
            res = bozo_amd.global_tension(s["Q"], s["K"], s["V"], scale, bias=s["bias"], W_local=case["Wl"] or None)
            out, tau = res if case["Wl"] else (res, None)
        else:
            res = bozo_amd.causal_tension(s["Q"], s["K"], s["V"], case["W"], scale, return_tau=case["tau"],
                                          bias=s["bias"], normalize=case["norm"])
            out, tau = res if case["tau"] else (res, None)
    if not case["grad"]:
        return {"out": out, "tau": tau}
    outs, into = ([out], [s["dOut"]]) if tau is None else ([out, tau], [s["dOut"], s["dTau"]])
    dQ, dK, dV = torch.autograd.grad(outs, [s["Q"], s["K"], s["V"]], into)
    return {"out": out, "tau": tau, "dQ": dQ, "dK": dK, "dV": dV}


# ------------------------------------------------------------------ work

def work(case):
    eq = _qk_dtype(case["flow"]).itemsize
    ev = _v_dtype(case["flow"]).itemsize
    if case["kind"] == "decode":
        rows = min(case["pos"], case["W"])
        per = case["N"] * case["H"] * case["D"]
        # the live rows of both caches, the new rows read and appended, q and out
        byts = per * (rows * (eq + ev) + 2 * (eq + ev) + 2 * eq)
        byts += case["N"] * case["H"] * case["W"] * eq if case["tau"] else 0
        return {"bytes": byts, "flops": 4 * per * (rows + int(case["self_key"]))}
    pairs, D = _pairs(case), case["D"]
    n = case["B"] * case["T"] * case["H"] * D
    if case["kind"] == "layer":
        dim, rows = case["H"] * D, case["B"] * case["T"]
        tau = case["B"] * case["T"] * case["H"] * case["W"] * 4
        # x, out, dout, dx in float32, tau and dtau, four weights and their gradients
        return {"bytes": 4 * 4 * n + 2 * tau + 2 * 4 * 4 * dim * dim,
                "flops": 12 * D * pairs + 4 * 6 * rows * dim * dim}
    width = case["W"] if case["kind"] == "window" else case["Wl"]
    tau = case["B"] * case["T"] * case["H"] * width * eq if (case["kind"] == "global" or case["tau"]) else 0
    bias = 4 * case["B"] * case["T"] * (width if case["kind"] == "window" else case["T"]) if case["bias"] else 0
    if not case["grad"]:
        return {"bytes": n * (3 * eq + ev) + tau + bias, "flops": 4 * D * pairs}
    # Q, K, V, dOut (dTau, bias) in; out, dQ, dK, dV (tau) out
    return {"bytes": n * (6 * eq + 2 * ev) + 2 * tau + bias, "flops": 12 * D * pairs}


# ------------------------------------------------------------------ tolerance

def tolerance(case):
    """About four times what changing the order of the sums shows.  bf16 and
    float16 results are rounded to their own type from float32 sums of products
    whose P and G factors are rounded too; with float32 rows the bf16 dV of the
    autocast flow is the coarsest output (a rounding that falls the other way)."""
    flow = case["flow"]
    if case["kind"] == "layer":
        return {"rel": 1.2e-2, "max": 0.3}
    if flow == "bf16":
        return {"rel": 1e-2, "max": 0.1}
    if flow == "f16":
        return {"rel": 1.5e-3, "max": 2e-2}
    if flow == "autocast":
        if case["kind"] == "decode" or not case["grad"]:
            return {"rel": 3e-6, "max": 3e-4}
        return {"rel": 1e-3, "max": 2e-2}
    return {"rel": 3e-6, "max": 3e-4}


# ------------------------------------------------------------------ 64 bits

def _mask(case, T):
    q = torch.arange(T, device="cuda")[:, None]
    k = torch.arange(T, device="cuda")[None, :]
    if case["kind"] == "global":
        return k <= q
    return (k < q) & (k >= q - case["W"])


def _slots(case, T):
    """(key index, whether it exists) of each tau slot, [T, width]."""
    q = torch.arange(T, device="cuda")[:, None]
    if case["kind"] == "global":
        key = T - 1 - torch.arange(case["Wl"], device="cuda")[None, :].expand(T, -1)
        return key, key <= q
    key = q - case["W"] + torch.arange(case["W"], device="cuda")[None, :]
    return key.clamp(min=0), key >= 0


def _one_sequence(case, q, k, v, bias):
    """out and tau of one sequence, [H, T, D] each, float64, all pairs at once."""
    T = q.shape[1]
    score = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(case["D"])
    if bias is not None:
        if case["kind"] == "global":
            score = score + bias
        else:  # [T, W] by slot: key s of query t is slot s - t + W
            slot = (torch.arange(T, device="cuda")[None, :] - torch.arange(T, device="cuda")[:, None] + case["W"])
            full = torch.gather(bias, 1, slot.clamp(0, case["W"] - 1))
            score = score + full
    p = torch.sigmoid(score) * _mask(case, T).to(score.dtype)
    out = torch.matmul(p, v)
    norm = case.get("norm", "mass")  # "raw": the sum as it is
    if norm == "mass":
        out = out / p.sum(-1, keepdim=True).clamp(min=1e-6)
    elif norm == "count":
        n = torch.arange(T, device="cuda").clamp(max=case["W"]).clamp(min=1).to(out.dtype)
        out = out / n[:, None]
    width = case.get("W") if case["kind"] != "global" else case["Wl"]
    if not width or not (case["kind"] == "global" or case.get("tau", True)):
        return out, None
    key, ok = _slots(case, T)
    tau = torch.gather(p, 2, key.expand(p.shape[0], -1, -1)) * ok.to(p.dtype)
    return out, tau


def _exact_op(case, s):
    rows = []
    for b in range(case["B"]):
        q, k, v = (s[n][b].detach().double().transpose(0, 1).contiguous().requires_grad_(case["grad"])
                   for n in ("Q", "K", "V"))
        with torch.set_grad_enabled(case["grad"]):
            out, tau = _one_sequence(case, q, k, v, None if s["bias"] is None else s["bias"][b].double())
        got = [out.detach(), None if tau is None else tau.detach()]
        if case["grad"]:
            outs, into = [out], [s["dOut"][b].double().transpose(0, 1)]
            if tau is not None:
                outs, into = outs + [tau], into + [s["dTau"][b].double().transpose(0, 1)]
            got += list(torch.autograd.grad(outs, [q, k, v], into))
        rows.append([None if x is None else x.transpose(0, 1) for x in got])
    full = [None if x[0] is None else torch.stack(list(x)) for x in zip(*rows)]
    return dict(zip(("out", "tau", "dQ", "dK", "dV"), full + [None] * (5 - len(full)) if case["grad"] else full))


def _exact_decode(case, s):
    q, kc, vc = s["q"].double(), s["k_cache"].double(), s["v_cache"].double()
    W, pos = case["W"], case["pos"]
    live = min(pos, W)
    p = torch.sigmoid((kc * q[:, :, None]).sum(-1) / math.sqrt(case["D"]))
    p = p * (torch.arange(W, device="cuda") < live).to(p.dtype)
    num, mass, keys = (p[..., None] * vc).sum(2), p.sum(-1), live
    if case["self_key"]:
        own = torch.sigmoid((s["k_new"].double() * q).sum(-1) / math.sqrt(case["D"]))
        num, mass, keys = num + own[..., None] * s["v_new"].double(), mass + own, keys + 1
    if case["norm"] == "mass":
        num = num / mass.clamp(min=1e-6)[..., None]
    elif case["norm"] == "count":
        num = num / max(keys, 1)
    tau = None
    if case["tau"]:  # slot w, oldest first
        tau = torch.gather(p, 2, ((torch.arange(W, device="cuda") + pos) % W).expand_as(p))
    return {"out": num, "tau": tau, "k_cache": None, "v_cache": None, "pos": None}


def _exact_layer(case, s):
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    x = s["x"].detach().double().requires_grad_(True)
    w = {n: t.double().requires_grad_(True) for n, t in s["weights"].items()}
    scale = s["norm_scale"].double().requires_grad_(True)
    half = D // 2
    inv = 1.0 / (10_000 ** (torch.arange(half, dtype=torch.float32, device="cuda") / half))
    ang = torch.arange(T, dtype=torch.float32, device="cuda")[:, None] * inv[None, :]
    cos, sin = ang.cos().double()[:, None], ang.sin().double()[:, None]

    def turn(z):
        a, b = z[..., :half], z[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    q, k, v = ((x @ w[n].t()).view(B, T, H, D) for n in ("wq", "wk", "wv"))
    q, k = turn(q), turn(k)
    per = [_one_sequence(dict(case, tau=True), *(z[b].transpose(0, 1) for z in (q, k, v)), None) for b in range(B)]
    msg = torch.stack([p[0].transpose(0, 1) for p in per]).reshape(B, T, H * D)
    tau = torch.stack([p[1].transpose(0, 1) for p in per])
    y = x + msg @ w["wo"].t()
    out = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * scale
    grads = torch.autograd.grad([out, tau], [x] + [w[n] for n in ("wq", "wk", "wv", "wo")] + [scale],
                                [s["dout"].double(), s["dtau"].double()])
    return {"out": out.detach(), "tau": tau.detach(), "grads": list(grads)}


def exact(case, seed):
    """What ``run`` returns for these inputs, in 64 bits, from plain torch."""
    s = _inputs(case, seed)
    if case["kind"] == "decode":
        return _exact_decode(case, s)
    if case["kind"] == "layer":
        return _exact_layer(case, s)
    return _exact_op(case, s)
