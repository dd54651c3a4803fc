"""The calls whose speed is measured: what a program that uses CVMM has it do.

Two kinds of case:

- ``proj``: one training step of one projection (selector from the router's
  ids, forward, backward to the input, the experts' weights and, for a
  weighted selection, the routing weights).  ``mode`` "up" takes token rows
  and returns one row per route; "down" takes one row per route and returns
  the weighted sum per token.  ``heads`` > 0 routes per attention head, two
  of the head's own experts each (SwitchHead's value and output projections).
- ``ffn``: a whole MoE feed-forward block (router projection, top-k router,
  up projection + GELU, weighted down projection), as inference (``train``
  False: decode with a few tokens, prefill with many) or as a training step
  with every gradient.

``op`` is the compute type: "float32" runs without autocast, the 16-bit types
under it.  ``weights`` is the type the expert weights are kept in: float32
master weights in training, and those or bfloat16 weights in inference.
"""
import math

import torch

import cvmm_codex_amd as cvmm

_TYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _proj(name, mode, tokens, d_in, d_out, experts, k, op, heads=0):
    case = {"kind": "proj", "mode": mode, "tokens": tokens, "d_in": d_in, "d_out": d_out, "experts": experts,
            "k": k, "op": op, "heads": heads}
    return {"name": name, **case} if name else case


def _ffn(name, tokens, d_model, d_expert, experts, k, op, weights, skew, train):
    case = {"kind": "ffn", "tokens": tokens, "d_model": d_model, "d_expert": d_expert, "experts": experts, "k": k,
            "op": op, "weights": weights, "skew": skew, "train": train}
    return {"name": name, **case} if name else case


def listed():
    return [
        # the smallest step: a unit-sized fp32 layer, all launches and host work
        _proj("tiny_fp32", "up", 512, 256, 64, 16, 4, "float32"),
        # sampling a few sequences from a model in training (float32 master weights under autocast)
        _ffn("decode_4", 4, 1024, 128, 64, 8, "bfloat16", "float32", 0.0, False),
        # one decode step of a served batch, weights kept in bfloat16
        _ffn("decode_32", 32, 2048, 512, 128, 8, "bfloat16", "bfloat16", 0.0, False),
        # prefill of one prompt of odd length
        _ffn("prefill_1999", 1999, 2048, 512, 128, 8, "bfloat16", "bfloat16", 0.5, False),
        # training in float32 (the op's own default without autocast)
        _proj("up_fp32", "up", 4096, 1024, 128, 64, 8, "float32"),
        # widths and a batch that no tile divides, as a model sized to a parameter budget has
        _proj("up_odd", "up", 4095, 412, 130, 63, 8, "bfloat16"),
        # few wide experts, two per token, under float16 autocast
        _proj("up_wide_fp16", "up", 4096, 1024, 4096, 8, 2, "float16"),
        # the MoE feed-forward projections at their usual training size
        _proj("up_1024", "up", 8192, 1024, 128, 64, 8, "bfloat16"),
        _proj("down_1024", "down", 8192, 128, 1024, 64, 8, "bfloat16"),
        # SwitchHead value and output projections
        _proj("switch_v_2048", "up", 8192, 2048, 64, 256, 64, "bfloat16", 32),
        _proj("switch_o_2048", "down", 8192, 64, 2048, 256, 64, "bfloat16", 32),
        # the largest: a whole feed-forward block's training step with a skewed router
        _ffn("ffn_train_2048", 16384, 2048, 512, 128, 8, "bfloat16", "float32", 1.1, True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    family = rng.choice(["fp32", "odd", "16bit", "16bit", "wide", "switch", "decode", "prefill", "train"])
    mode = rng.choice(["up", "down"])
    if family == "fp32":
        d_model, d_expert = 8 * _log_int(rng, 16, 128), 4 * _log_int(rng, 8, 48)
        tokens, experts, k = _log_int(rng, 256, 4096), _log_int(rng, 8, 64), rng.choice([1, 2, 4, 8])
        op, heads = "float32", 0
    elif family == "odd":
        d_model, d_expert = _log_int(rng, 200, 900), _log_int(rng, 40, 260)
        tokens, experts, k = _log_int(rng, 500, 6000), _log_int(rng, 8, 128), rng.choice([2, 4, 8])
        op, heads = rng.choice(["bfloat16", "float16"]), 0
    elif family == "16bit":
        d_model, d_expert = 8 * _log_int(rng, 32, 256), 8 * _log_int(rng, 8, 64)
        tokens, experts, k = _log_int(rng, 512, 8192), _log_int(rng, 8, 128), rng.choice([1, 2, 4, 8])
        op, heads = rng.choice(["bfloat16", "bfloat16", "float16"]), 0
    elif family == "wide":
        d_model, d_expert = 64 * _log_int(rng, 8, 32), 64 * _log_int(rng, 16, 64)
        tokens, experts, k = _log_int(rng, 1024, 6000), rng.choice([4, 8, 16]), rng.choice([1, 2])
        op, heads = rng.choice(["bfloat16", "float16"]), 0
    elif family == "switch":
        heads, per_head = rng.choice([8, 16, 32]), rng.choice([4, 5, 8])
        d_model, d_expert = 64 * _log_int(rng, 8, 32), rng.choice([64, 80, 96, 128])
        tokens, experts, k = _log_int(rng, 512, 5000), heads * per_head, 2 * heads
        op = "bfloat16"
    else:
        d_model, d_expert = 64 * _log_int(rng, 8, 32), 64 * _log_int(rng, 2, 8)
        experts, k, op = _log_int(rng, 8, 128), rng.choice([2, 4, 8]), rng.choice(["bfloat16", "bfloat16", "float16"])
        train = family == "train"
        lo, hi = {"decode": (1, 64), "prefill": (200, 4000), "train": (1000, 8000)}[family]
        weights = "float32" if train else rng.choice(["float32", op])
        return _ffn("", _log_int(rng, lo, hi), d_model, d_expert, experts, k, op, weights,
                    rng.choice([0.0, 0.5, 1.1]), train)
    d_in, d_out = (d_model, d_expert) if mode == "up" else (d_expert, d_model)
    return _proj("", mode, tokens, d_in, d_out, experts, k, op, heads)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _routing(case, g):
    """(ids [T, k] int64, gates [T, k] float32) as a softmax router picks them."""
    T, E, k, heads = case["tokens"], case["experts"], case["k"], case["heads"]
    if heads:
        gates, ids = torch.softmax(_randn(g, T, heads, E // heads), dim=-1).topk(2, dim=-1)
        ids = ids + (E // heads) * torch.arange(heads, device="cuda").view(1, heads, 1)
        return ids.reshape(T, k), gates.reshape(T, k)
    # mild differences between the experts' loads, as a balanced router shows
    gates, ids = torch.softmax(_randn(g, T, E) + 0.3 * _randn(g, E), dim=-1).topk(k, dim=-1)
    return ids.contiguous(), gates.contiguous()


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    op = _TYPES[case["op"]]
    T, E, k = case["tokens"], case["experts"], case["k"]
    state = {"case": case}
    if case["kind"] == "proj":
        d_in, d_out = case["d_in"], case["d_out"]
        ids, gates = _routing(case, g)
        state["sel"] = ids
        state["keys"] = (_randn(g, E, d_in, d_out) / math.sqrt(d_in)).requires_grad_()
        if case["mode"] == "up":
            state["x"] = _randn(g, T, d_in).to(op).requires_grad_()
            state["grad"] = _randn(g, T, k, d_out).to(op)
        else:
            state["x"] = torch.nn.functional.gelu(_randn(g, T, k, d_in)).to(op).requires_grad_()
            state["gates"] = gates.requires_grad_()
            state["grad"] = _randn(g, T, d_out).to(op)
        return state
    D, H = case["d_model"], case["d_expert"]
    train, kept = case["train"], _TYPES[case["weights"]]
    state["x"] = _randn(g, 1, T, D).to(op).requires_grad_(train)
    state["gate"] = (_randn(g, D, E) / math.sqrt(D)).to(kept).requires_grad_(train)
    # a router that prefers some experts: log of a Zipf law over them
    ranks = torch.arange(1, E + 1, device="cuda", dtype=torch.float32)
    state["bias"] = torch.log_softmax(-case["skew"] * torch.log(ranks), dim=0)
    state["w_up"] = (_randn(g, E, D, H) / math.sqrt(D)).to(kept).requires_grad_(train)
    state["w_down"] = (_randn(g, E, H, D) / math.sqrt(H)).to(kept).requires_grad_(train)
    if train:
        state["grad"] = _randn(g, 1, T, D).to(op)
    return state


def _autocast(op):
    return torch.autocast("cuda", dtype=_TYPES[op] if op != "float32" else torch.bfloat16, enabled=op != "float32")


def _block(state):
    case, x = state["case"], state["x"]
    logits = cvmm.cvmm_gate_logits(x, state["gate"]) + state["bias"]
    weights, _, sel_up = cvmm.cvmm_route_topk(logits, case["k"], True)
    hidden = cvmm.cvmm_gelu(x, sel_up, state["w_up"])
    sel_down = cvmm.cvmm_prepare_sel2(sel_up, weights, route_input=True)
    return cvmm.cvmm(hidden, sel_down, state["w_down"])


def run(state):
    case = state["case"]
    if case["kind"] == "ffn":
        if not case["train"]:
            with torch.no_grad(), _autocast(case["op"]):
                return {"y": _block(state)}
        with _autocast(case["op"]):
            y = _block(state)
        names = ["x", "gate", "w_up", "w_down"]
    else:
        up = case["mode"] == "up"
        with _autocast(case["op"]):
            sel = cvmm.cvmm_prepare_sel2(state["sel"], None if up else state["gates"], route_input=not up)
            y = cvmm.cvmm(state["x"], sel, state["keys"])
        names = ["x", "keys"] if up else ["x", "keys", "gates"]
    grads = torch.autograd.grad(y, [state[n] for n in names], state["grad"])
    return {"y": y.detach(), **{"grad_" + n: v for n, v in zip(names, grads)}}


def work(case):
    """Inputs once, outputs once, and the products' multiply-adds.  (An
    inference block reads the weights of the experts that its routes can
    reach at most.)"""
    T, E, k = case["tokens"], case["experts"], case["k"]
    a = 4 if case["op"] == "float32" else 2
    R = T * k
    if case["kind"] == "proj":
        d_in, d_out = case["d_in"], case["d_out"]
        in_rows, out_rows = (T, R) if case["mode"] == "up" else (R, T)
        nbytes = 2 * a * (in_rows * d_in + out_rows * d_out) + 8 * E * d_in * d_out + 8 * R
        if case["mode"] == "down":
            nbytes += 8 * R
        return {"bytes": nbytes, "flops": 6 * R * d_in * d_out}
    D, H = case["d_model"], case["d_expert"]
    wb = 4 if case["weights"] == "float32" else 2
    if case["train"]:
        return {"bytes": 4 * a * T * D + 2 * wb * (D * E + 2 * E * D * H),
                "flops": 6 * (2 * R * D * H + T * D * E)}
    return {"bytes": 2 * a * T * D + wb * (D * E + 2 * min(E, R) * D * H), "flops": 2 * (2 * R * D * H + T * D * E)}


def tolerance(case):
    """About four times the error against 64 bits that is measured: sums in
    another order in fp32; in 16 bits each operand's and result's rounding
    (two to three of them in one projection, five in a block)."""
    rel = {"float32": 1e-5, "bfloat16": 1.2e-2, "float16": 2e-3}[case["op"]]
    return {"rel": rel if case["kind"] == "proj" else 1.7 * rel}


def _experts64(rows, ids, keys):
    """rows[r] @ keys[ids[r]] in float64, expert by expert."""
    order = torch.argsort(ids, stable=True)
    parts = torch.split(rows.index_select(0, order), torch.bincount(ids, minlength=keys.shape[0]).tolist())
    out = torch.cat([p @ keys[e] for e, p in enumerate(parts)])
    return out.index_select(0, torch.argsort(order))


def exact(case, seed):
    state = prepare(case, seed)
    T, k = case["tokens"], case["k"]
    leaf = {n: v.detach().double().requires_grad_() for n, v in state.items()
            if isinstance(v, torch.Tensor) and v.is_floating_point() and n not in ("grad", "bias")}
    if case["kind"] == "proj":
        ids = state["sel"].reshape(-1)
        if case["mode"] == "up":
            rows = leaf["x"].repeat_interleave(k, dim=0)
            y = _experts64(rows, ids, leaf["keys"]).view(T, k, -1)
            names = ["x", "keys"]
        else:
            y = _experts64(leaf["x"].reshape(T * k, -1), ids, leaf["keys"]).view(T, k, -1)
            y = (y * leaf["gates"].unsqueeze(-1)).sum(1)
            names = ["x", "keys", "gates"]
    else:
        op = _TYPES[case["op"]]
        x = leaf["x"].reshape(T, -1)
        logits = x @ leaf["gate"]
        # the router reads logits rounded to the compute type: the choice of experts follows from those
        with torch.no_grad():
            rounded = (x @ leaf["gate"].to(op).double()).to(op).double() + state["bias"].double()
            ids = torch.sort(rounded, dim=-1, descending=True, stable=True).indices[:, :k]
        probs = torch.softmax(logits + (rounded - logits).detach(), dim=-1).gather(1, ids)
        gates = probs / probs.sum(-1, keepdim=True)
        ids = ids.reshape(-1)
        hidden = torch.nn.functional.gelu(_experts64(x.repeat_interleave(k, dim=0), ids, leaf["w_up"]))
        y = _experts64(hidden, ids, leaf["w_down"]).view(T, k, -1)
        y = (y * gates.unsqueeze(-1)).sum(1).view(1, T, -1)
        names = ["x", "gate", "w_up", "w_down"]
        if not case["train"]:
            return {"y": y.detach()}
    grads = torch.autograd.grad(y, [leaf[n] for n in names], state["grad"].double())
    return {"y": y.detach(), **{"grad_" + n: v for n, v in zip(names, grads)}}
