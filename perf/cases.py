"""The calls that programs built on spider_moe_amd make, as measurable cases.

Three kinds of call:

  block   SpiderMoELayer.forward_loops / forward_loops_exit: all loops of the
          recurrent block in one call (router, edge messages, dispatch, expert
          FFN, LayerNorm), on the weights a program loads and packs once
  delta   sparse_expert_delta: the expert FFN alone, on routing that the
          caller already has
  ffn     ForgeGEMM.fp8_expert_ffn: one expert's FFN on fp8 weights, with the
          input in bf16 or quantized to fp8 on the way

Weights are N(0, 0.02), hidden states N(0, 1), as the seeded workloads of
spider_moe_amd.workloads; everything is drawn on the GPU from the seed alone.
exact() restates the same computation in 64 bits with plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "spider-web-moe_amd"))

LOOP_EMBED = 32
ALPHA, BETA, EPS = 0.5, 0.1, 1e-5

# The models of the cases: the benchmark's three block shapes and the default
# ModelConfig (which is fp32).
MODELS = {
    "swiglu16": dict(H=1024, E=16, K=2, M=2, U=2816, R=6, act="swiglu"),
    "gelu32": dict(H=1024, E=32, K=4, M=2, U=1408, R=4, act="gelu"),
    "gelu64": dict(H=2048, E=64, K=2, M=4, U=1408, R=4, act="gelu"),
    "default": dict(H=256, E=8, K=2, M=3, U=512, R=6, act="gelu"),
}


def _block(name, model, dtype, experts, tokens, *, skew=0.0, empty=0, exit=False):
    return {"name": name, "kind": "block", "model": model, "dtype": dtype, "experts": experts,
            "tokens": tokens, "skew": skew, "empty": empty, "exit": exit}


def listed():
    return [
        # one user's next token on the fp8 model: the smallest call, all latency
        _block("decode-1-fp8", "swiglu16", "bf16", "fp8", 1),
        # a full decode batch on the fp8 model: weight streaming
        _block("decode-64-fp8", "swiglu16", "bf16", "fp8", 64),
        # a ragged decode batch with the early-exit gate
        _block("decode-37-bf16-exit", "swiglu16", "bf16", "bf16", 37, exit=True),
        # a small decode batch on the wide int4 model
        _block("decode-16-int4", "gelu64", "bf16", "int4", 16),
        # one short prompt (or a decode batch past 64 users) on the fp8 model
        _block("chunk-200-fp8", "swiglu16", "bf16", "fp8", 200),
        # one ordinary prompt of odd length, bf16
        _block("prefill-777-bf16", "swiglu16", "bf16", "bf16", 777),
        # a large prefill batch (8 prompts of 2048)
        _block("prefill-16384-bf16", "swiglu16", "bf16", "bf16", 16384),
        # the same under Zipf-skewed routing with four experts empty
        _block("prefill-16384-skew", "gelu32", "bf16", "bf16", 16384, skew=1.2, empty=4),
        # decode tokens and a prefill chunk in one step, int4 experts
        _block("mixed-2176-int4", "gelu64", "bf16", "int4", 2176),
        # the default configuration in fp32, 4 prompts of 512
        _block("prefill-2048-f32", "default", "f32", "f32", 2048),
        # the expert FFN alone, called with routing from elsewhere
        {"name": "delta-2000-bf16", "kind": "delta", "dtype": "bf16", "tokens": 2000, "H": 1024,
         "U": 2816, "E": 16, "K": 2},
        # one expert's FFN with fp8 weights and a quantized input
        {"name": "ffn-4096-fp8", "kind": "ffn", "tokens": 4096, "H": 1024, "U": 2816,
         "quantize_input": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "chunk", "chunk", "prefill", "wide", "f32", "delta", "ffn"])
    if kind == "decode":
        model = rng.choice(["swiglu16", "swiglu16", "gelu64"])
        experts = "int4" if model == "gelu64" else rng.choice(["fp8", "bf16", "int4"])
        c = _block("", model, "bf16", experts, _log_int(rng, 1, 64), exit=rng.random() < 0.25)
    elif kind == "chunk":
        model = rng.choice(["swiglu16", "gelu32"])
        c = _block("", model, "bf16", rng.choice(["fp8", "bf16", "int4"]), _log_int(rng, 65, 4096))
    elif kind == "prefill":
        if rng.random() < 0.5:
            c = _block("", "swiglu16", "bf16", "bf16", _log_int(rng, 4096, 16384))
        else:
            c = _block("", "gelu32", "bf16", "bf16", _log_int(rng, 4096, 16384),
                       skew=round(rng.uniform(0.0, 1.2), 2), empty=rng.randrange(5))
    elif kind == "wide":
        c = _block("", "gelu64", "bf16", "int4", _log_int(rng, 65, 2176))
    elif kind == "f32":
        c = _block("", "default", "f32", "f32", _log_int(rng, 16, 4096))
    elif kind == "delta":
        h, u, e = rng.choice([(1024, 2816, 16), (1024, 1408, 32), (256, 512, 8)])
        c = {"kind": "delta", "dtype": "bf16", "tokens": _log_int(rng, 16, 4096), "H": h, "U": u,
             "E": e, "K": rng.choice([1, 2, 4])}
    else:
        h, u = rng.choice([(1024, 2816), (1024, 1408), (2048, 1408), (1000, 2800)])
        c = {"kind": "ffn", "tokens": _log_int(rng, 64, 8192), "H": h, "U": u,
             "quantize_input": rng.random() < 0.7}
    c.pop("name", None)
    return c


# ------------------------------------------------------------- inputs ----
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.bfloat16


def _normal(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)


def _block_params(case, seed):
    """The layer's state dict, and the inputs h and x0 [N, 1, H]."""
    m, dt, gen = MODELS[case["model"]], _dtype(case), _generator(seed)
    h, e, u, r = m["H"], m["E"], m["U"], m["R"]
    bias = torch.zeros(r, e, device="cuda")
    if case["skew"] or case["empty"]:
        perm = torch.randperm(e, generator=gen, device="cuda")
        rank = torch.empty(e, device="cuda")
        rank[perm] = torch.arange(1, e + 1, device="cuda", dtype=torch.float32)
        bias = bias - case["skew"] * rank.log()
        if case["empty"]:
            bias[:, perm[e - case["empty"]:]] = -1e4
    p = {
        "loop_bias": bias.to(dt),
        "router.weight": _normal(gen, e, h, std=0.02, dtype=dt),
        "loop_embedding.weight": _normal(gen, r, LOOP_EMBED, std=0.02, dtype=dt),
        "edge_generator.weight": _normal(gen, e * e, h + LOOP_EMBED, std=0.02, dtype=dt),
        "edge_generator.bias": torch.zeros(e * e, device="cuda", dtype=dt),
        "norm.weight": torch.ones(h, device="cuda", dtype=dt),
        "norm.bias": torch.zeros(h, device="cuda", dtype=dt),
        "exit_head.weight": _normal(gen, 1, h, std=0.02, dtype=dt),
        "exit_head.bias": torch.zeros(1, device="cuda", dtype=dt),
    }
    for i in range(e):
        p[f"edge_value.{i}.weight"] = _normal(gen, h, h, std=0.02, dtype=dt)
        p[f"experts.{i}.0.weight"] = _normal(gen, 2 * u if m["act"] == "swiglu" else u, h, std=0.02,
                                             dtype=dt)
        p[f"experts.{i}.2.weight"] = _normal(gen, h, u, std=0.02, dtype=dt)
        if m["act"] == "gelu":
            p[f"experts.{i}.0.bias"] = _normal(gen, u, std=0.02, dtype=dt)
            p[f"experts.{i}.2.bias"] = _normal(gen, h, std=0.02, dtype=dt)
    n = case["tokens"]
    return p, _normal(gen, n, 1, h, dtype=dt), _normal(gen, n, 1, h, dtype=dt)


def _delta_inputs(case, seed):
    gen, dt = _generator(seed), _dtype(case)
    n, h, u, e, k = (case[x] for x in ("tokens", "H", "U", "E", "K"))
    logits = torch.randn(n, e, generator=gen, device="cuda")
    w, idx = logits.softmax(-1).topk(k, dim=-1)
    w = w / w.sum(-1, keepdim=True)
    return dict(messages=_normal(gen, 1, n, h, dtype=dt), top_indices=idx.view(1, n, k),
                top_weights=w.view(1, n, k), w_up=_normal(gen, e, u, h, std=0.02, dtype=dt),
                b_up=_normal(gen, e, u, std=0.02, dtype=dt),
                w_down=_normal(gen, e, h, u, std=0.02, dtype=dt),
                b_down=_normal(gen, e, h, std=0.02, dtype=dt))


def _ffn_inputs(case, seed):
    gen, dt = _generator(seed), torch.bfloat16
    n, h, u = case["tokens"], case["H"], case["U"]
    return (_normal(gen, n, h, dtype=dt), _normal(gen, u, h, std=0.02, dtype=dt),
            _normal(gen, u, std=0.02, dtype=dt), _normal(gen, h, u, std=0.02, dtype=dt),
            _normal(gen, h, std=0.02, dtype=dt))


# -------------------------------------------------------- the program ----
def prepare(case, seed):
    if case["kind"] == "delta":
        return case, _delta_inputs(case, seed)
    if case["kind"] == "ffn":
        from spider_moe_amd.forge import ForgeConfig, ForgeGEMM
        return case, ForgeGEMM(ForgeConfig(gemm_fp8=True)), _ffn_inputs(case, seed)
    from spider_moe_amd import SpiderMoELayer
    from spider_moe_amd.config import ModelConfig
    m = MODELS[case["model"]]
    params, h, x0 = _block_params(case, seed)
    cfg = ModelConfig(vocab_size=64, hidden_size=m["H"], num_experts=m["E"], top_k=m["K"],
                      edges_per_expert=m["M"], num_loops=m["R"], expert_ffn_size=m["U"],
                      loop_embed_size=LOOP_EMBED, expert_activation=m["act"], expert_parallel=False)
    with torch.device("meta"):
        layer = SpiderMoELayer(cfg)
    layer.load_state_dict(params, assign=True)
    layer.eval().requires_grad_(False)
    if case["experts"] == "fp8":
        layer.quantize_experts_fp8()
    elif case["experts"] == "int4":
        layer.quantize_experts(group_size=128, scale_dtype=torch.float16)
    layer.workspace_bytes(case["tokens"])  # lays the weights out, as at a server's start
    return case, layer, h, x0


def run(state):
    case = state[0]
    if case["kind"] == "delta":
        from spider_moe_amd import sparse_expert_delta
        return sparse_expert_delta(**state[1], num_experts=case["E"], top_k=case["K"],
                                   expert_parallel=False)
    if case["kind"] == "ffn":
        x, w_up, b_up, w_down, b_down = state[2]
        return state[1].fp8_expert_ffn(x, w_up, b_up, w_down, b_down,
                                       quantize_input=case["quantize_input"])
    _, layer, h, x0 = state
    with torch.no_grad():
        if case["exit"]:
            return layer.forward_loops_exit(h, x0)
        return layer.forward_loops(h, x0)


# --------------------------------------------------------------- work ----
def work(case):
    n = case["tokens"]
    if case["kind"] == "delta":
        h, u, e, k = (case[x] for x in ("H", "U", "E", "K"))
        touched = e * (1 - (1 - k / e) ** n)
        return {"bytes": touched * 2 * (2 * h * u + h + u) + n * (2 * 2 * h + 12 * k),
                "flops": 4.0 * n * k * h * u}
    if case["kind"] == "ffn":
        h, u = case["H"], case["U"]
        return {"bytes": 2 * 2 * h * u + 2 * (h + u) + 2 * 2 * n * h, "flops": 4.0 * n * h * u}
    m = MODELS[case["model"]]
    h, e, k, em, u, r = (m[x] for x in ("H", "E", "K", "M", "U", "R"))
    swiglu = m["act"] == "swiglu"
    size = 4 if case["dtype"] == "f32" else 2
    per_weight = {"f32": 4.0, "bf16": 2.0, "fp8": 1.0, "int4": 0.5 + 2 / 128}[case["experts"]]
    live = e - case["empty"]
    dests = e * (1 - (1 - em / e) ** min(k, live))  # distinct destinations of a token
    # experts and destinations that a pass touches, tokens routing alike in every loop
    experts = live * (1 - (1 - k / live) ** n)
    touched = e * (1 - (1 - dests / e) ** n)
    flops = n * r * (2.0 * h * e + 2.0 * (h + LOOP_EMBED) * e * k + 2.0 * h * h * dests
                     + (6.0 if swiglu else 4.0) * h * u * k)
    read = (experts * per_weight * (3 if swiglu else 2) * h * u + touched * size * h * h
            + size * (h * e + (h + LOOP_EMBED) * e * min(e, n * k)))
    return {"bytes": read + 3 * size * n * h, "flops": flops}


def tolerance(case):
    """About four times what the path differs from the same steps in plain
    torch with the same roundings (bf16 messages, activations, expert outputs
    and block state) and sums in another order.

    In a bf16 block a sum in another order turns a near-tie of the router or
    of an edge now and then (0.1% of the tokens over all loops), and such a
    token is off by a tenth or more: measured rel 4e-3 to 5e-3 over thousands
    of tokens, 1e-2 where one token of a decode batch turns and over the wide
    int4 model, and 0.5 of the root mean square at a single value."""
    if case["kind"] != "block":
        return {"rel": 1e-2}
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    many = case["tokens"] >= 512 and case["model"] != "gelu64"
    return {"rel": 0.02 if many else 0.03, "max": 0.99}


# -------------------------------------------------------------- exact ----
def _fp8_values(w, per_row):
    """The values of e4m3 codes with one scale per output row (or one in all)."""
    w = w.float()
    amax = w.abs().amax(-1, keepdim=True) if per_row else w.abs().amax()
    scale = (amax / 448.0).clamp_min(1e-12)
    return (w / scale).to(torch.float8_e4m3fn).double() * scale.double()


def _int4_values(w, group=128):
    rows, k = w.shape
    g = group if k % group == 0 else k
    w = w.float().view(rows, k // g, g)
    scale = w.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 7.0
    q = torch.round(w / scale).clamp(-8, 7)
    return (q.double() * scale.half().double()).view(rows, k)


def _expert_weight(case, w):
    if case["experts"] == "fp8":
        return _fp8_values(w, per_row=True)
    if case["experts"] == "int4":
        return _int4_values(w)
    return w


def _linear(x, w, b=None):
    return F.linear(x, w.to(x.dtype), None if b is None else b.to(x.dtype))


def _block_loops(case, params, h, x0, dtype=torch.float64, stored=lambda t: t):
    """All loops in `dtype`; `stored` is applied where values go back to memory."""
    m = MODELS[case["model"]]
    e, k, em, u, swiglu = m["E"], m["K"], m["M"], m["U"], m["act"] == "swiglu"
    n = case["tokens"]
    p = {name: t.to(dtype) for name, t in params.items()
         if not name.startswith(("experts.", "edge_value."))}
    h, x0 = h.view(n, -1).to(dtype), x0.view(n, -1).to(dtype)
    live = torch.ones(n, dtype=torch.bool, device="cuda")
    for r in range(m["R"]):
        probs = (_linear(h, p["router.weight"]) + p["loop_bias"][r]).softmax(-1)
        top_w, top_i = probs.topk(k, dim=-1)
        top_w = top_w / top_w.sum(-1, keepdim=True).clamp_min(1e-9)
        # messages: every selected source's em strongest edges, by destination
        coef = torch.zeros(n, e, dtype=dtype, device="cuda")
        emb = p["loop_embedding.weight"][r].expand(n, -1)
        logits = _linear(torch.cat([h, emb], -1), p["edge_generator.weight"], p["edge_generator.bias"])
        logits = logits.view(n, e, e).gather(1, top_i.unsqueeze(-1).expand(n, k, e))
        values, dest = logits.topk(em, dim=-1)
        coef.scatter_add_(1, dest.reshape(n, k * em), values.softmax(-1).reshape(n, k * em))
        msg = torch.zeros_like(h)
        for d in range(e):
            rows = (coef[:, d] > 0).nonzero().squeeze(-1)
            if rows.numel():
                y = _linear(h[rows], params[f"edge_value.{d}.weight"]) * coef[rows, d:d + 1]
                msg.index_add_(0, rows, stored(y))
        msg = stored(msg)
        delta = torch.zeros_like(h)
        for x in range(e):
            rows, slot = (top_i == x).nonzero(as_tuple=True)
            if rows.numel():
                up = _linear(msg[rows], _expert_weight(case, params[f"experts.{x}.0.weight"]),
                             params.get(f"experts.{x}.0.bias"))
                a = F.silu(up[:, :u]) * up[:, u:] if swiglu else F.gelu(up)
                y = _linear(stored(a), _expert_weight(case, params[f"experts.{x}.2.weight"]),
                            params.get(f"experts.{x}.2.bias"))
                delta.index_add_(0, rows, stored(y * top_w[rows, slot].unsqueeze(-1)))
        new = F.layer_norm(h + ALPHA * delta + BETA * x0, (m["H"],), p["norm.weight"], p["norm.bias"], EPS)
        h = torch.where(live.unsqueeze(-1), stored(new), h)
        if case["exit"]:
            live = live & ~(_linear(h, p["exit_head.weight"], p["exit_head.bias"]).squeeze(-1).sigmoid() > 0.85)
    return h.view(n, 1, m["H"])


def exact(case, seed):
    if case["kind"] == "delta":
        t = _delta_inputs(case, seed)
        n, k = case["tokens"], case["K"]
        x = t["messages"].view(n, -1).double()
        idx, w = t["top_indices"].view(n, k), t["top_weights"].view(n, k).double()
        out = torch.zeros_like(x)
        for e in range(case["E"]):
            rows, slot = (idx == e).nonzero(as_tuple=True)
            a = F.gelu(_linear(x[rows], t["w_up"][e], t["b_up"][e]))
            out.index_add_(0, rows, _linear(a, t["w_down"][e], t["b_down"][e]) * w[rows, slot].unsqueeze(-1))
        return out.view(1, n, -1)
    if case["kind"] == "ffn":
        x, w_up, b_up, w_down, b_down = _ffn_inputs(case, seed)
        x = _fp8_values(x, per_row=False) if case["quantize_input"] else x.double()
        a = F.gelu(_linear(x, _fp8_values(w_up, per_row=False), b_up))
        return _linear(a, _fp8_values(w_down, per_row=False), b_down)
    params, h, x0 = _block_params(case, seed)
    out = _block_loops(case, params, h, x0)
    return (out, None, None) if case["exit"] else out
