"""Test helpers: seeded cases, oracle comparisons, and the stated tolerance.

Tolerance (north star): max|out - ref| <= 2e-2 * RMS(ref), with ref the exact (fp64) value of
the op on the same bf16 inputs. op_eager itself rounds to bf16 after every stage and sits
~5-8% of RMS away from that exact value at these shapes, so against op_eager the reference's own
gate is used: allclose(out, op_eager, atol=2e-2, rtol=2e-2)
(src/configs/registry/cohere2_moe_experts.py:89-92).
"""

from __future__ import annotations

import torch

from oracle import eager as O

TOL_RMS = 2e-2


def rand_case(seed, T, H, Fi, E, K, layout="concat", act="silu", bias=False, std=0.02, invalid=0, skew=0.0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, H, generator=g).bfloat16()
    if layout == "concat":
        W1 = (torch.randn(E, 2 * Fi, H, generator=g) * std).bfloat16()
        W2 = (torch.randn(E, H, Fi, generator=g) * std).bfloat16()
    else:
        W1 = (torch.randn(E, H, 2 * Fi, generator=g) * std).bfloat16()
        W2 = (torch.randn(E, Fi, H, generator=g) * std).bfloat16()
    b1 = (torch.randn(E, 2 * Fi, generator=g) * std).bfloat16() if bias else None
    b2 = (torch.randn(E, H, generator=g) * std).bfloat16() if bias else None
    logits = torch.randn(T, E, generator=g)
    if skew > 0:
        logits = logits + skew * torch.log(torch.arange(1, E + 1, dtype=torch.float32)).neg()
    probs = torch.softmax(logits, -1)
    w, idx = torch.topk(probs, K, dim=-1)
    w = (w / w.sum(-1, keepdim=True)).bfloat16()
    for i in range(invalid):
        t, k = int(torch.randint(T, (1,), generator=g)), int(torch.randint(K, (1,), generator=g))
        idx[t, k] = E + i if i % 2 == 0 else -1 - i
    return dict(x=x, idx=idx, w=w, W1=W1, W2=W2, b1=b1, b2=b2, layout=layout, act=act)


def oracle_fp64(c, rows=None):
    sel = slice(None) if rows is None else rows
    return O.experts_fp64(c["x"][sel], c["idx"][sel], c["w"][sel], c["W1"], c["W2"], c["b1"], c["b2"],
                          layout=c["layout"], act=c["act"])


def oracle_eager(c, rows=None):
    sel = slice(None) if rows is None else rows
    return O.experts_eager(c["x"][sel], c["idx"][sel], c["w"][sel], c["W1"], c["W2"], c["b1"], c["b2"],
                           layout=c["layout"], act=c["act"])


def run_gpu(c, device, decode=False, dev_tensors=None):
    from cernels_amd import ops

    d = dev_tensors or to_device(c, device)
    layout = ops.LAYOUT_CONCAT if c["layout"] == "concat" else ops.LAYOUT_INTERLEAVED
    act = ops.ACT_SILU if c["act"] == "silu" else ops.ACT_GPTOSS
    return ops.moe_experts(d["x"], d["W1"], d["W2"], d["idx"], d["w"], d["idx"].shape[1], layout=layout, act=act,
                           gate_up_bias=d["b1"], down_bias=d["b2"], decode=decode)


def packed_form(T, H, Fi, E, K, act="silu"):
    """Which kernels a packed call of these sizes takes (``_native.PACKED_FORMS``); act: "silu", "gptoss" or a megablocks
    act_id. Tests of one form assert it, so that a moved line cannot turn them into tests of another."""
    from cernels_amd import _native, ops

    a = {"silu": ops.ACT_SILU, "gptoss": ops.ACT_GPTOSS, **ops.MEGABLOCKS_ACTS}[act]
    form = _native.lib().cernels_moe_experts_packed_form(T, H, Fi, E, K, a)
    assert form >= 0, (T, H, Fi, E, K, act)
    return _native.PACKED_FORMS[form]


def form_of(c):
    """``packed_form`` of a case of ``rand_case``."""
    (E, n1, n2), (T, H), K = c["W1"].shape, c["x"].shape, c["idx"].shape[1]
    return packed_form(T, H, (n1 if c["layout"] == "concat" else n2) // 2, E, K, c["act"])


def to_device(c, device):
    mv = lambda t, dt=None: None if t is None else (t.to(dt) if dt else t).contiguous().to(device)  # noqa: E731
    return dict(x=mv(c["x"]), W1=mv(c["W1"]), W2=mv(c["W2"]), idx=mv(c["idx"], torch.int32),
                w=mv(c["w"], torch.float32), b1=mv(c["b1"], torch.float32), b2=mv(c["b2"], torch.float32))


def half_ulp_bf16(ref64: torch.Tensor) -> torch.Tensor:
    """Half the bf16 spacing at each reference value: the error of correctly rounding it to bf16."""
    a = ref64.abs().clamp_min(2.0 ** -126)
    return torch.exp2(torch.floor(torch.log2(a)) - 8)


def assert_within_tolerance(out, ref64, what="", strict=False):
    """|out - ref| <= 2e-2*RMS(ref) + half a bf16 ulp of ref, elementwise.

    The output is bf16, so even a correctly rounded result is up to half an ulp away from the
    exact value; at the 6-8*RMS outliers of these workloads that alone is 0.012-0.016*RMS. The
    bar therefore bounds the error beyond the output's own rounding by 2e-2*RMS. ``strict`` also
    demands max|out - ref| <= 2e-2*RMS with no allowance.
    """
    out64, ref64 = out.double().cpu(), ref64.double().cpu()
    st = O.error_stats(out64, ref64)
    excess = ((out64 - ref64).abs() - half_ulp_bf16(ref64)).max().item() if ref64.numel() else 0.0
    st["excess_ratio"] = excess / st["rms_ref"] if st["rms_ref"] > 0 else 0.0
    assert excess <= TOL_RMS * st["rms_ref"], (
        f"{what}: max(|err| - ulp/2)={excess:.3e} > {TOL_RMS}*RMS({st['rms_ref']:.3e}); max|err|={st['max_abs']:.3e}")
    if strict:
        assert st["ratio"] <= TOL_RMS, f"{what}: max|err|={st['max_abs']:.3e} > {TOL_RMS}*RMS({st['rms_ref']:.3e})"
    return st


def assert_reference_verify(out, eager, what=""):
    ok = torch.allclose(out.float().cpu(), eager.float().cpu(), atol=2e-2, rtol=2e-2)
    assert ok, f"{what}: fails the reference's allclose(atol=rtol=2e-2) against op_eager"


# ---- whole-output strict bar at full BASELINE / reference sizes ----------------------------------------

_FULL_CASES: dict = {}


def full_case(name, device):
    """(case on the CPU, its device tensors, the exact fp64 output on the device) of a BASELINE or reference
    workload, built once per process. The exact value is the float64 restatement (the oracle, a checker
    only) computed on the GPU in float64."""
    hit = _FULL_CASES.get(name)
    if hit is not None:
        return hit
    from cernels_amd.configs.registry import BASELINE_SHAPES, REFERENCE_SHAPES
    from cernels_amd.configs.synth import make_inputs, make_weights

    s = BASELINE_SHAPES.get(name) or REFERENCE_SHAPES[name]
    print(f"[full case {name}] generating", flush=True)
    inp, wts = make_inputs(s), make_weights(s)
    c = dict(x=inp.x, idx=inp.top_k_index, w=inp.top_k_weights, W1=wts.gate_up_proj, W2=wts.down_proj,
             b1=wts.gate_up_proj_bias, b2=wts.down_proj_bias, layout=s.layout, act=s.act)
    d = to_device(c, device)
    print(f"[full case {name}] fp64 oracle on the GPU", flush=True)
    mv = lambda t: None if t is None else t.to(device)  # noqa: E731
    ref = O.experts_fp64(mv(c["x"]), mv(c["idx"]), mv(c["w"]), mv(c["W1"]), mv(c["W2"]), mv(c["b1"]), mv(c["b2"]),
                         layout=s.layout, act=s.act)
    _FULL_CASES.clear()  # one workload resident at a time
    _FULL_CASES[name] = (c, d, ref)
    return c, d, ref


def assert_strict_full(out, ref, what=""):
    """The north-star bar on a whole output, with no allowance: max|out - exact| <= 2e-2 * RMS(exact), or the
    correctly rounded answer bf16(exact)'s own max error where that is larger (no bf16 output can do better;
    it happens on the reference's deepseek routing, whose weights are not renormalised). Returns
    (error, floor, bar), each relative to RMS(exact)."""
    out = out.to(ref.device).double()
    rms = float(ref.pow(2).mean().sqrt())
    err = float((out - ref).abs().max()) / rms
    floor = float((ref.to(torch.bfloat16).double() - ref).abs().max()) / rms
    bar = max(TOL_RMS, floor)
    print(f"[strict {what}] max|err|/RMS = {err:.6f} (correctly rounded bf16: {floor:.6f}; bar {bar:.6f})",
          flush=True)
    assert err <= bar, f"{what}: max|err| = {err:.6f} RMS > {bar:.6f} RMS (bf16(exact) reads {floor:.6f})"
    return err, floor, bar
