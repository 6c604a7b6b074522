"""The calls that are timed when the layer's speed is looked at, with their inputs and float64 results.

Three public entry points are covered: ``dsmoe.DeepSeekMoE`` (the layer, forward and training step, fp32 and bf16,
and fp32 parameters under bf16 autocast), ``dsmoe.grouped_moe_dispatch`` (the operator seam) and
``dsmoe.mla.triton_mla_attention`` (the attention operator).  Shapes are those of tests/_cases.py, bench.py and the
model configurations the tests cite, with token counts from a single decoded token to a full training step.

``listed()`` are the named cases and ``draw(rng)`` gives another one of the same ranges.  ``prepare`` makes inputs,
``run`` does one pass, ``exact`` gives the pass's results in float64 from plain torch, ``work`` the bytes and
operations a pass cannot do without, ``tolerance`` the error that the data types of a pass leave."""
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "deepseek-v3-lite_amd"))
import dsmoe  # noqa: E402
from dsmoe.mla import triton_mla_attention  # noqa: E402

# Layer shapes: dim, routed experts, top-k, expert width, shared experts, shared width.
LAYERS = {
    "tiny": dict(D=64, E=4, k=2, I=128, S=1, Is=128),           # tests/_cases.py C0
    "422m": dict(D=768, E=20, k=4, I=384, S=1, Is=384),         # configs/pretrain_a100_422m.yaml:20-28
    "single": dict(D=1024, E=16, k=4, I=512, S=1, Is=1024),     # tests/_cases.py C1
    "wide": dict(D=2048, E=64, k=6, I=1408, S=2, Is=1408),      # tests/_cases.py C3, C4
}
# Attention shapes: heads, latent rank, q/k width without and with rotary part, value width.
MLAS = {
    "small": dict(H=4, R=16, Dn=16, Dr=16, Dv=16),              # configs/pretrain_1650_2m.yaml:14-26
    "422m": dict(H=12, R=192, Dn=48, Dr=24, Dv=64),             # configs/pretrain_a100_422m.yaml:22-34
}


def _layer(shape, T, mode, train):
    """mode: "fp32" and "bf16" (parameters and activations), "autocast" (fp32 parameters, bf16 autocast)."""
    return dict(kind="layer", shape=shape, T=T, mode=mode, train=train)


def _grouped(shape, rows, skew, train):
    return dict(kind="grouped", shape=shape, T=rows, skew=skew, train=train)


def _mla(shape, B, S_q, S_kv, train):
    return dict(kind="mla", shape=shape, B=B, S_q=S_q, S_kv=S_kv, train=train)


def listed():
    return [
        # the small pretraining configuration, whose layers run in fp32: a forward of 8 x 128 tokens
        dict(name="layer_fp32_tiny_fwd", **_layer("tiny", 1024, "fp32", False)),
        # a full-precision training step on one sequence of the larger configuration
        dict(name="layer_fp32_422m_train", **_layer("422m", 2048, "fp32", True)),
        # generating one token for one user: the weights of the experts it touches
        dict(name="layer_bf16_wide_decode1", **_layer("wide", 1, "bf16", False)),
        # generating for 64 users at once: every expert's weights
        dict(name="layer_bf16_wide_decode64", **_layer("wide", 64, "bf16", False)),
        # a short prompt, or a large decode batch: a few ragged rows for each expert
        dict(name="layer_bf16_wide_prompt333", **_layer("wide", 333, "bf16", False)),
        # prefill of 8192 tokens: the headline workload of bench.py
        dict(name="layer_bf16_wide_prefill", **_layer("wide", 8192, "bf16", False)),
        # the training step of bench.py
        dict(name="layer_bf16_wide_train", **_layer("wide", 16384, "bf16", True)),
        # the trainer's own form: fp32 parameters under bf16 autocast, one micro batch of two sequences less some padding
        dict(name="layer_autocast_422m_train", **_layer("422m", 4001, "autocast", True)),
        # the operator seam in training, rows already sorted, uneven experts and an empty one
        dict(name="grouped_bf16_single_train", **_grouped("single", 3000, 1.0, True)),
        # one generated token for each of 8 users over their cached context
        dict(name="mla_422m_decode", **_mla("422m", 8, 1, 1537, False)),
        # a second chunk of a prompt after a cached first one
        dict(name="mla_422m_chunk", **_mla("422m", 1, 500, 1300, False)),
        # attention of the training step: micro batch 8, full sequences
        dict(name="mla_422m_train", **_mla("422m", 8, 2048, 2048, True)),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "grouped", "mla", "mla", "mla"])
    if kind == "layer":
        mode = rng.choice(["fp32", "bf16", "bf16", "autocast"])
        train = rng.random() < 0.5
        if mode == "fp32":
            return _layer(rng.choice(["tiny", "422m"]), _log_int(rng, 16, 2048), mode, train)
        if mode == "autocast":
            return _layer(rng.choice(["422m", "single"]), _log_int(rng, 64, 16384), mode, train)
        if train:
            return _layer(rng.choice(["422m", "single", "wide"]), _log_int(rng, 64, 16384), mode, train)
        return _layer(rng.choice(["422m", "single", "wide", "wide"]), _log_int(rng, 1, 8192), mode, train)
    if kind == "grouped":
        return _grouped(rng.choice(["422m", "single"]), _log_int(rng, 32, 8192), rng.choice([0.0, 1.0]), rng.random() < 0.5)
    shape = rng.choice(["small", "422m", "422m"])
    form = rng.choice(["decode", "chunk", "train"])
    if form == "decode":
        return _mla(shape, _log_int(rng, 1, 32), 1, _log_int(rng, 16, 2048), False)
    if form == "chunk":
        S_kv = _log_int(rng, 32, 2048)
        return _mla(shape, rng.choice([1, 1, 2, 4]), _log_int(rng, 2, S_kv), S_kv, False)
    S = _log_int(rng, 128, 2048)
    return _mla(shape, rng.choice([1, 2, 4, 8]), S, S, True)


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _dtype(case):
    return torch.bfloat16 if case.get("mode") == "bf16" or case["kind"] == "grouped" else torch.float32


def _normal(g, std, dtype, *shape):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _layer_inputs(case, seed):
    """x ~ N(0, 1), weights ~ N(0, 0.02), gate bias ~ N(0, 0.01), the upstream gradient ~ N(0, 1).  Under autocast x
    and the gradient are fp32 tensors of values that a bf16 layer before and after has produced, so that the layer's
    own cast of x does not change which experts a token goes to."""
    s, g, dt = LAYERS[case["shape"]], _gen(seed), _dtype(case)
    sd = {"gate.weight": _normal(g, 0.02, torch.float32, s["E"], s["D"]), "gate.bias": _normal(g, 0.01, torch.float32, s["E"])}
    for group, n, width in (("experts", s["E"], s["I"]), ("shared_experts", s["S"], s["Is"])):
        for e in range(n):
            sd[f"{group}.{e}.w1.weight"] = _normal(g, 0.02, dt, width, s["D"])
            sd[f"{group}.{e}.w2.weight"] = _normal(g, 0.02, dt, s["D"], width)
            sd[f"{group}.{e}.w3.weight"] = _normal(g, 0.02, dt, width, s["D"])
    x = _normal(g, 1.0, dt, case["T"], s["D"])
    dy = _normal(g, 1.0, dt, case["T"], s["D"]) if case["train"] else None
    if case["mode"] == "autocast":
        x, dy = x.bfloat16().float(), dy.bfloat16().float() if case["train"] else None
    return sd, x, dy


def _group_rows(case, seed):
    """Rows of each expert: uneven by weights 1 / (1 + skew i), one expert without rows."""
    E = LAYERS[case["shape"]]["E"]
    w = [1.0 / (1.0 + case["skew"] * i) for i in range(E)]
    w[int(seed) % E] = 0.0
    rows = [int(case["T"] * v / sum(w)) for v in w]
    rows[max(range(E), key=lambda i: w[i])] += case["T"] - sum(rows)
    return rows


def _grouped_inputs(case, seed):
    s, g, dt = LAYERS[case["shape"]], _gen(seed), _dtype(case)
    w1 = _normal(g, 0.02, dt, s["E"], s["I"], s["D"])
    w2 = _normal(g, 0.02, dt, s["E"], s["D"], s["I"])
    w3 = _normal(g, 0.02, dt, s["E"], s["I"], s["D"])
    x = _normal(g, 1.0, dt, case["T"], s["D"])
    sw = torch.rand(case["T"], generator=g, device="cuda").to(dt)
    dy = _normal(g, 1.0, dt, case["T"], s["D"]) if case["train"] else None
    offsets = torch.tensor([0] + _group_rows(case, seed), dtype=torch.int64).cumsum(0).cuda()
    return x, w1, w2, w3, sw, offsets, dy


def _mla_inputs(case, seed):
    """Queries in bf16.  In training the layer hands over fp32 latent rows and views of its fp32 weight under bf16
    autocast (dsmoe/mla.py); a bf16 model at inference has everything in bf16."""
    s, g, B = MLAS[case["shape"]], _gen(seed), case["B"]
    dt = torch.float32 if case["train"] else torch.bfloat16
    q_nope = _normal(g, 1.0, torch.bfloat16, B, s["H"], case["S_q"], s["Dn"])
    q_pe = _normal(g, 1.0, torch.bfloat16, B, s["H"], case["S_q"], s["Dr"])
    ctx_kv = _normal(g, 1.0, dt, B, case["S_kv"], s["R"])
    ctx_pe = _normal(g, 1.0, dt, B, case["S_kv"], s["Dr"])
    wkv_b = _normal(g, 0.1, dt, s["H"] * (s["Dn"] + s["Dv"]), s["R"])
    dout = _normal(g, 1.0, torch.bfloat16, B, case["S_q"], s["H"], s["Dv"]) if case["train"] else None
    return q_nope, q_pe, ctx_kv, ctx_pe, wkv_b, dout


def prepare(case, seed):
    st = {"case": case}
    if case["kind"] == "layer":
        s = LAYERS[case["shape"]]
        sd, x, dy = _layer_inputs(case, seed)
        with torch.device("meta"):
            m = dsmoe.DeepSeekMoE({"dim": s["D"], "n_routed_experts": s["E"], "n_shared_experts": s["S"], "moe_inter_dim": s["I"],
                                   "n_activated_experts": s["k"], "shared_inter_dim": s["Is"]})
        m.load_state_dict(sd, assign=True)
        m.train(case["train"])
        named = dict(m.named_parameters())
        st.update(m=m, x=x.requires_grad_(case["train"]), dy=dy, params=list(named.values()),
                  returned=[named[n] for n in _returned(case, seed)])
    elif case["kind"] == "grouped":
        x, w1, w2, w3, sw, off, dy = _grouped_inputs(case, seed)
        st.update(off=off, dy=dy, leaves=[t.requires_grad_(case["train"]) for t in (x, w1, w2, w3, sw)])
    else:
        *ts, dout = _mla_inputs(case, seed)
        st.update(dout=dout, leaves=[t.requires_grad_(case["train"]) for t in ts])
    return st


# ---------------------------------------------------------------------------- one pass
def _returned(case, seed):
    """The weights whose gradients a pass returns: all of them, of routed experts at most 17 spread over the layer,
    others for another seed (the caller takes a bounded number of outputs)."""
    s = LAYERS[case["shape"]]
    n = min(s["E"], 17)
    experts = sorted({(int(seed) + i * s["E"] // n) % s["E"] for i in range(n)})
    return ["gate.weight"] + [f"{grp}.{e}.{w}.weight" for grp, ids in (("experts", experts), ("shared_experts", range(s["S"])))
                              for e in ids for w in ("w1", "w2", "w3")]


def _head_views(w, s):
    """The key and value up-projections of each head: views of the one weight, as models/mla.py:127-129 takes them."""
    w = w.view(s["H"], s["Dn"] + s["Dv"], s["R"])
    return w[:, :s["Dn"]], w[:, s["Dn"]:]


def _run_layer(st):
    case, m, x = st["case"], st["m"], st["x"]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=case["mode"] == "autocast"):
        if not case["train"]:
            with torch.no_grad():
                return [m(x), m._last_indices, m._last_weights]
        for t in (x, *st["params"]):
            t.grad = None
        y = m(x)
    y.backward(st["dy"])
    return [y.detach(), m._last_indices, m._last_weights, x.grad, *[p.grad for p in st["returned"]]]


def _run_grouped(st):
    x, w1, w2, w3, sw = leaves = st["leaves"]
    if not st["case"]["train"]:
        with torch.no_grad():
            return [dsmoe.grouped_moe_dispatch(x, w1, w2, w3, sw, st["off"])]
    for t in leaves:
        t.grad = None
    y = dsmoe.grouped_moe_dispatch(x, w1, w2, w3, sw, st["off"])
    y.backward(st["dy"])
    return [y.detach(), *[t.grad for t in leaves]]


def _run_mla(st):
    case, (q_nope, q_pe, ctx_kv, ctx_pe, wkv_b) = st["case"], st["leaves"]
    s = MLAS[case["shape"]]
    scale = (s["Dn"] + s["Dr"]) ** -0.5
    q_start = case["S_kv"] - case["S_q"]
    if not case["train"]:
        with torch.no_grad():
            return [triton_mla_attention(q_nope, q_pe, ctx_kv, ctx_pe, *_head_views(wkv_b, s), scale, True, q_start)]
    for t in st["leaves"]:
        t.grad = None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = triton_mla_attention(q_nope, q_pe, ctx_kv, ctx_pe, *_head_views(wkv_b, s), scale, True, q_start)
    out.backward(st["dout"])
    return [out.detach(), *[t.grad for t in st["leaves"]]]


def run(state):
    return {"layer": _run_layer, "grouped": _run_grouped, "mla": _run_mla}[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    if case["kind"] == "mla":
        s, B, Sq, Skv = MLAS[case["shape"]], case["B"], case["S_q"], case["S_kv"]
        pairs = B * s["H"] * (Sq * (Skv - Sq) + Sq * (Sq + 1) // 2)
        keys, queries = B * s["H"] * Skv, B * s["H"] * Sq
        heads = keys * 2 * s["R"] * (s["Dn"] + s["Dv"]) + pairs * 2 * (s["Dn"] + s["Dr"] + s["Dv"])
        latent = queries * 2 * s["R"] * (s["Dn"] + s["Dv"]) + pairs * 2 * (2 * s["R"] + s["Dr"])
        w = 4 if case["train"] else 2
        kv = (B * Skv * (s["R"] + s["Dr"]) + s["H"] * (s["Dn"] + s["Dv"]) * s["R"]) * w
        q, out = queries * (s["Dn"] + s["Dr"]) * 2, queries * s["Dv"] * 2
        if not case["train"]:
            return {"bytes": kv + q + out, "flops": min(heads, latent)}
        return {"bytes": 2 * (kv + q + out), "flops": 3 * min(heads, latent)}
    s, T = LAYERS[case["shape"]], case["T"]
    w = 2 if _dtype(case) == torch.bfloat16 else 4
    if case["kind"] == "grouped":
        weights = 3 * s["E"] * s["I"] * s["D"] * w
        flops = 6 * T * s["I"] * s["D"]
    else:
        touched = s["E"] * (1 - (1 - s["k"] / s["E"]) ** T)
        weights = 3 * s["D"] * (touched * s["I"] + s["S"] * s["Is"]) * w + 4 * s["E"] * s["D"]
        flops = 6 * s["D"] * T * (s["k"] * s["I"] + s["S"] * s["Is"]) + 2 * T * s["E"] * s["D"]
    rows = T * s["D"] * w
    if not case["train"]:
        return {"bytes": weights + 2 * rows, "flops": flops}
    return {"bytes": 2 * weights + 4 * rows, "flops": 3 * flops}


def tolerance(case):
    """About four times the error against exact() that was measured over listed() and drawn cases: relative 3e-7
    (tiny) to 1.1e-6 in fp32, 3.0e-3 in a bf16 layer's forward and 3.5e-3 in its gradients, 4.5e-3 under autocast,
    2.7e-3 in attention and 5.0e-3 in its gradients.  A token whose choice of experts is a near tie may take the other
    expert ("differ"), which moves its whole row, so the layer states no largest error."""
    if case["kind"] == "layer":
        if case["mode"] == "fp32":
            return {"rel": 4e-6, "differ": 1e-3}
        return {"rel": 1.8e-2 if case["mode"] == "autocast" else 1.4e-2, "differ": 1e-3}
    if case["kind"] == "grouped":
        return {"rel": 1.4e-2, "max": 0.2} if case["train"] else {"rel": 1e-2, "max": 6e-2}
    return {"rel": 2e-2, "max": 0.4} if case["train"] else {"rel": 1e-2, "max": 4e-2}


# ---------------------------------------------------------------------------- float64 results
def _swiglu(x, w1, w2, w3):
    return (torch.nn.functional.silu(x @ w1.T) * (x @ w3.T)) @ w2.T


def _exact_layer(case, seed):
    s = LAYERS[case["shape"]]
    sd, x, dy = _layer_inputs(case, seed)
    names = ["gate.weight"] + [f"{grp}.{e}.{w}.weight" for grp, n in (("experts", s["E"]), ("shared_experts", s["S"]))
                               for e in range(n) for w in ("w1", "w2", "w3")]
    p = {n: sd[n].double().requires_grad_(case["train"]) for n in names}
    x = x.double().requires_grad_(case["train"])
    with torch.set_grad_enabled(case["train"]):
        scores = torch.sigmoid(x @ p["gate.weight"].T)
        idx = (scores + sd["gate.bias"].double()).topk(s["k"], dim=-1)[1]
        w = scores.gather(1, idx)
        w = w / w.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(s["E"]):
            t, j = (idx == e).nonzero(as_tuple=True)
            if t.numel():
                o = _swiglu(x[t], *[p[f"experts.{e}.{n}.weight"] for n in ("w1", "w2", "w3")])
                y = y.index_add(0, t, o * w[t, j].unsqueeze(1))
        for e in range(s["S"]):
            y = y + _swiglu(x, *[p[f"shared_experts.{e}.{n}.weight"] for n in ("w1", "w2", "w3")])
    out = [y.detach(), idx, w.detach()]
    if case["train"]:
        wanted = [x, *[p[n] for n in _returned(case, seed)]]
        gr = torch.autograd.grad(y, wanted, dy.double(), allow_unused=True)
        out += [g if g is not None else torch.zeros_like(t) for g, t in zip(gr, wanted)]
    return out


def _exact_grouped(case, seed):
    x, w1, w2, w3, sw, off, dy = _grouped_inputs(case, seed)
    leaves = [t.double().requires_grad_(case["train"]) for t in (x, w1, w2, w3, sw)]
    x, w1, w2, w3, sw = leaves
    off = off.tolist()
    with torch.set_grad_enabled(case["train"]):
        y = torch.cat([_swiglu(x[a:b], w1[e], w2[e], w3[e]) for e, (a, b) in enumerate(zip(off, off[1:]))]) * sw.unsqueeze(1)
    if not case["train"]:
        return [y]
    return [y.detach(), *torch.autograd.grad(y, leaves, dy.double())]


def _exact_mla(case, seed):
    s = MLAS[case["shape"]]
    *ts, dout = _mla_inputs(case, seed)
    outs, grads = [], []
    wkv = ts[4].double().requires_grad_(case["train"])
    wk, wv = _head_views(wkv, s)
    Sq, Skv = case["S_q"], case["S_kv"]
    mask = torch.arange(Skv, device="cuda")[None, :] > torch.arange(Sq, device="cuda")[:, None] + (Skv - Sq)
    for b in range(case["B"]):
        leaves = [t[b].double().requires_grad_(case["train"]) for t in ts[:4]]
        with torch.set_grad_enabled(case["train"]):
            qn, qp, c, pe = leaves
            kn, v = c @ wk.transpose(1, 2), c @ wv.transpose(1, 2)
            z = (qn @ kn.transpose(1, 2) + qp @ pe.T) * (s["Dn"] + s["Dr"]) ** -0.5
            o = (z.masked_fill(mask, float("-inf")).softmax(-1) @ v).transpose(0, 1)
        outs.append(o.detach())
        if case["train"]:
            grads.append(torch.autograd.grad(o, [*leaves, wkv], dout[b].double(), retain_graph=True))
    if not case["train"]:
        return [torch.stack(outs)]
    per_input = list(zip(*grads))
    return [torch.stack(outs), *[torch.stack(g) for g in per_input[:4]], sum(per_input[4])]


def exact(case, seed):
    return {"layer": _exact_layer, "grouped": _exact_grouped, "mla": _exact_mla}[case["kind"]](case, seed)
