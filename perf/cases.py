"""The work a user of this framework has it do, one routed-experts layer at a time, through the public entry points.

A program that runs a mixture-of-experts model calls one of these entries once per layer and step:

* ``cohere2`` / ``deepseek`` (``cernels_amd.kops.registry.<slug>_moe_experts``): the experts of a decoder layer, with the
  router outside. ``kernel`` for prompts (weights packed once per module), ``decode_kernel`` while generating.
* ``gpt_oss`` / ``qwen3_next`` / ``megablocks``: a whole MoE block from the hidden states, router inside the call (and the
  gated shared expert for qwen3-next). The same entry serves prompts and generation.
* ``stored`` (``cernels_amd.ops.moe_experts``): prompts on the weights as the checkpoint stores them, for callers that
  keep no packed copy.

Sizes are those of ``cernels_amd.configs.registry`` (the layers' shapes and prompt lengths); drawn cases vary the number of
tokens over the whole range, and the layer's shape in part of them.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from cernels_amd import ops
from cernels_amd.configs import modules as M
from cernels_amd.kops.registry import (_packed, cohere2_moe_experts, deepseek_ocr2_moe_experts, gpt_oss_moe_experts,
                                       megablocks_moe, qwen3_next_moe_experts)

DEV = "cuda"
STD = 0.02  # weights ~ N(0, 0.02), hidden states ~ N(0, 1), as the benchmark configurations draw them

# hidden, expert intermediate, experts, top-k of each layer
SHAPES = {
    "deepseek": (1280, 896, 64, 6),
    "cohere2": (2048, 768, 128, 8),
    "gpt_oss": (2880, 2880, 32, 4),
    "qwen3_next": (2048, 512, 512, 10),
    "megablocks": (2048, 5632, 8, 2),
}
SHARED_FFN = 512  # qwen3-next's shared expert
# kind -> the layers it serves
KINDS = {
    "decode": ("cohere2", "deepseek"),
    "prefill": ("cohere2", "deepseek"),
    "block": ("gpt_oss", "qwen3_next", "megablocks"),
    "stored": ("cohere2", "deepseek", "gpt_oss"),
}


def _case(name, kind, layer, tokens, skew=0.0, shape=None):
    h, f, e, k = shape or SHAPES[layer]
    c = {"kind": kind, "layer": layer, "tokens": tokens, "hidden": h, "ffn": f, "experts": e, "top_k": k, "skew": skew}
    return {"name": name, **c} if name else c


def listed():
    return [
        # generating for one user: one token per step and layer
        _case("cohere2_decode_1", "decode", "cohere2", 1),
        # generating for a few users at once
        _case("deepseek_decode_8", "decode", "deepseek", 8),
        # a serving batch of generating users, an odd number of them
        _case("cohere2_decode_29", "decode", "cohere2", 29),
        # a short prompt (or one chunk of a long one): a few ragged rows per expert
        _case("cohere2_prefill_333", "prefill", "cohere2", 333),
        # whole prompts, the benchmark's lengths
        _case("deepseek_prefill_2048", "prefill", "deepseek", 2048),
        _case("cohere2_prefill_2048", "prefill", "cohere2", 2048),
        # gpt-oss layer, router in the call: one generated token, and the benchmark's prompt (the largest work here)
        _case("gpt_oss_block_1", "block", "gpt_oss", 1),
        _case("gpt_oss_block_4096", "block", "gpt_oss", 4096),
        # qwen3-next layer, router and shared expert in the call: three generating users, and a prompt whose routing is as
        # uneven as real routers' (expert popularity falls off as Zipf 1.2, the benchmark's skew)
        _case("qwen3_next_block_3", "block", "qwen3_next", 3),
        _case("qwen3_next_block_4096", "block", "qwen3_next", 4096, skew=1.2),
        # non-gated experts (GELU), few and wide
        _case("megablocks_block_4096", "block", "megablocks", 4096),
        # a prompt on the weights as stored, for callers that keep no packed copy
        _case("deepseek_stored_1000", "stored", "deepseek", 1000),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "prefill", "prefill", "block", "block", "block", "stored"))
    layer = rng.choice(KINDS[kind])
    h, f, e, k = SHAPES[layer]
    if rng.random() < 0.4:  # another layer of the same make
        h = 64 * rng.randint(8, 45)
        f = 64 * _log_int(rng, 6, 45)
        e = _log_int(rng, 8, 256)
        e = max(8, min(e, 1_600_000_000 // (6 * h * f)))  # no more weights, and below no more work, than the largest above
        k = rng.randint(1, 8)
    if kind == "decode":
        tokens = rng.randint(1, min(64, 256 // k))
    elif kind == "block":
        tokens = _log_int(rng, 1, 4096)
    else:
        tokens = _log_int(rng, 65, 2048)
    tokens = min(tokens, 800_000_000_000 // (6 * h * f * k))
    skew = rng.choice((0.0, 1.2)) if layer == "qwen3_next" else 0.0
    return _case(None, kind, layer, tokens, skew, (h, f, e, k))


def _normal(g, *shape, std=1.0):
    """N(0, std) in bf16, drawn in pieces so that no float32 copy of a whole weight is held."""
    out = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    flat = out.view(-1)
    step = 1 << 27
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        part.copy_(torch.randn(part.numel(), generator=g, device=DEV).mul_(std))
    return out


def _tensors(case, seed):
    """Everything of a case that is drawn: hidden states, weights and, where the router is the caller's, its choice."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    T, H, Fi, E, K = (case[n] for n in ("tokens", "hidden", "ffn", "experts", "top_k"))
    layer = case["layer"]
    d = {"x": _normal(g, T, H)}
    if layer == "gpt_oss":  # [E, H, 2F] with gate and up columns interleaved, [E, F, H], and biases
        d["w1"], d["w2"] = _normal(g, E, H, 2 * Fi, std=STD), _normal(g, E, Fi, H, std=STD)
        d["b1"], d["b2"] = _normal(g, E, 2 * Fi, std=STD), _normal(g, E, H, std=STD)
    elif layer == "megablocks":
        d["w1"], d["w2"] = _normal(g, E, H, Fi, std=STD), _normal(g, E, Fi, H, std=STD)
    else:
        d["w1"], d["w2"] = _normal(g, E, 2 * Fi, H, std=STD), _normal(g, E, H, Fi, std=STD)
    if case["kind"] == "block":
        d["router"] = _normal(g, E, H, std=STD)
        if layer == "gpt_oss":
            d["router_bias"] = _normal(g, E, std=STD)
        if case["skew"]:  # one feature that all tokens share carries each expert's popularity
            rank = torch.randperm(E, generator=g, device=DEV).double() + 1.0
            d["x"][:, 0] = 4.0
            d["router"][:, 0] = (-case["skew"] / 4.0 * torch.log(rank)).bfloat16()
        if layer == "qwen3_next":
            d["shared"] = (_normal(g, SHARED_FFN, H, std=STD), _normal(g, SHARED_FFN, H, std=STD),
                           _normal(g, H, SHARED_FFN, std=STD), _normal(g, 1, H, std=STD))
    else:
        logits = torch.randn(T, E, generator=g, device=DEV)
        if layer == "cohere2":  # top-k of the logits, sigmoid
            v, idx = torch.topk(logits, K, dim=-1)
            w = torch.sigmoid(v)
        elif layer == "deepseek":  # softmax, top-k
            w, idx = torch.topk(torch.softmax(logits, dim=-1), K, dim=-1)
        else:  # top-k, softmax
            v, idx = torch.topk(logits, K, dim=-1)
            w = torch.softmax(v, dim=-1)
        d["idx"], d["w"] = idx, w.bfloat16()  # int64 and bf16, as a transformers router hands them over
    return d


def _param(t):
    return torch.nn.Parameter(t, requires_grad=False)


def prepare(case, seed):
    d = _tensors(case, seed)
    kind, layer, H, E, K = case["kind"], case["layer"], case["hidden"], case["experts"], case["top_k"]
    s = {"kind": kind, "layer": layer, "top_k": K}
    with torch.no_grad():
        if kind == "stored":
            s.update(x=d["x"], w1=d["w1"], w2=d["w2"], idx=d["idx"].to(torch.int32), w=d["w"].float(), more={})
            if layer == "gpt_oss":
                s["more"] = {"layout": ops.LAYOUT_INTERLEAVED, "act": ops.ACT_GPTOSS, "gate_up_bias": d["b1"].float(),
                             "down_bias": d["b2"].float()}
        elif kind in ("decode", "prefill"):
            s.update(x=d["x"], idx=d["idx"], w=d["w"], module=M.Experts(d["w1"], d["w2"]))
            if kind == "prefill":
                _packed.packed_experts(s["module"])  # once per layer, when the model is loaded
        elif layer == "gpt_oss":
            router = M.GptOssRouter(H, E, K)
            router.weight, router.bias = _param(d["router"]), _param(d["router_bias"])
            s.update(x=d["x"][None], module=M.GptOssMlp(router, M.Experts(d["w1"], d["w2"], d["b1"], d["b2"])))
            gpt_oss_moe_experts._weights(s["module"].experts)
        elif layer == "qwen3_next":
            gate = M.Qwen3NextRouter(H, E, K)
            gate.weight = _param(d["router"])
            shared, sgate = M.DenseMlp(H, 1), torch.nn.Linear(H, 1, bias=False)
            g, u, dn, sg = d["shared"]
            shared.gate_proj.weight, shared.up_proj.weight, shared.down_proj.weight = _param(g), _param(u), _param(dn)
            sgate.weight = _param(sg)
            s.update(x=d["x"][None], module=M.Qwen3NextBlock(gate, M.Experts(d["w1"], d["w2"]), shared, sgate))
            _packed.packed_block(s["module"])
        else:
            args = M.MegablocksArgs(H, case["ffn"], E, K)
            router = M.MegablocksRouter(args)
            router.layer.weight = _param(d["router"])
            mlp = M.MegablocksMlp(d["w1"], d["w2"])
            s.update(x=d["x"], module=M.MegablocksMoe(router, M.MegablocksExperts(args, mlp)))
            _packed.packed_megablocks(mlp, ops.MEGABLOCKS_ACTS[megablocks_moe.act_id_of(args)])
    return s


def run(state):
    kind, layer, x = state["kind"], state["layer"], state["x"]
    if kind == "decode":
        f = cohere2_moe_experts if layer == "cohere2" else deepseek_ocr2_moe_experts
        return f.decode_kernel(x, state["idx"], state["w"], state["module"])
    if kind == "prefill":
        f = cohere2_moe_experts if layer == "cohere2" else deepseek_ocr2_moe_experts
        return f.kernel(x, state["idx"], state["w"], state["module"])
    if kind == "stored":
        return ops.moe_experts(x, state["w1"], state["w2"], state["idx"], state["w"], state["top_k"], **state["more"])
    if layer == "gpt_oss":
        return gpt_oss_moe_experts.kernel(x, state["module"])
    if layer == "qwen3_next":
        return qwen3_next_moe_experts.kernel(x, state["module"])
    return megablocks_moe.kernel(x, state["module"])


def _distinct(case):
    """Expected number of distinct experts that the tokens choose."""
    T, E, K = case["tokens"], case["experts"], case["top_k"]
    if not case["skew"]:
        return E * (1.0 - (1.0 - K / E) ** T)
    p = [r ** -case["skew"] for r in range(1, E + 1)]
    z = sum(p)
    return sum(1.0 - (1.0 - v / z) ** (T * K) for v in p)


def work(case):
    T, H, Fi, E, K = (case[n] for n in ("tokens", "hidden", "ffn", "experts", "top_k"))
    layer, block = case["layer"], case["kind"] == "block"
    mats = 2 if layer == "megablocks" else 3
    weights = _distinct(case) * (mats * H * Fi + (2 * Fi + H if layer == "gpt_oss" else 0)) * 2
    moved = weights + 2 * T * H * 2 + (E * H * 2 if block else T * K * 10)
    flops = 2 * mats * T * K * H * Fi + (2 * T * E * H if block else 0)
    if layer == "qwen3_next" and block:
        moved += 3 * H * SHARED_FFN * 2
        flops += 6 * T * H * SHARED_FFN
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    """bf16 results. The largest differences are those of a rounding to the next bf16 value (2^-8 of the value) and, in the
    decode entry, of the bf16 intermediate. Where the router is in the call, a logit next to a rounding boundary may
    change a token's last expert for one of almost the same logit: few tokens, whole rows."""
    if case["kind"] == "block":
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 5e-2}


def _route_exact(case, d):
    """The blocks' routers: logits as bf16 values, experts by logit (lower id first among equals), weights in bf16."""
    K, layer = case["top_k"], case["layer"]
    z = d["x"].double() @ d["router"].double().T
    if layer == "gpt_oss":
        z = z + d["router_bias"].double()
    z = z.bfloat16().double()
    v, idx = torch.sort(z, dim=-1, descending=True, stable=True)
    v, idx = v[:, :K], idx[:, :K]
    if layer == "gpt_oss":
        w = torch.softmax(v, dim=-1)
    else:
        w = torch.gather(torch.softmax(z, dim=-1), 1, idx)
        if layer == "qwen3_next":
            w = w / w.sum(dim=-1, keepdim=True)
    return idx, w.bfloat16()


def exact(case, seed):
    d = _tensors(case, seed)
    layer, E = case["layer"], case["experts"]
    idx, w = (d["idx"], d["w"]) if "idx" in d else _route_exact(case, d)
    x, w = d["x"].double(), w.double()
    out = torch.zeros_like(x)
    for e in range(E):
        t, k = torch.where(idx == e)
        if not t.numel():
            continue
        if layer == "megablocks":
            y = F.gelu(x[t] @ d["w1"][e].double(), approximate="tanh") @ d["w2"][e].double()
        elif layer == "gpt_oss":
            gu = x[t] @ d["w1"][e].double() + d["b1"][e].double()
            gate, up = gu[:, ::2].clamp(max=7.0), gu[:, 1::2].clamp(-7.0, 7.0)
            y = ((up + 1.0) * gate * torch.sigmoid(1.702 * gate)) @ d["w2"][e].double() + d["b2"][e].double()
        else:
            gate, up = (x[t] @ d["w1"][e].double().T).chunk(2, dim=-1)
            y = (F.silu(gate) * up) @ d["w2"][e].double().T
        out.index_add_(0, t, y * w[t, k, None])
    if "shared" in d:
        g, u, dn, sg = (v.double() for v in d["shared"])
        s = torch.sigmoid((x @ sg.T).bfloat16().double()).bfloat16().double()
        out += s * ((F.silu(x @ g.T) * (x @ u.T)) @ dn.T)
    return out[None] if case["kind"] == "block" and layer != "megablocks" else out
