"""Few rows per expert on packed weights: the streaming forms of moe_experts_packed, against the fp64 oracle.

Up to 32 tokens and 512 pairs the kernels route by themselves while the ids that their workgroups read stay few (up to 16
pairs with the sum over slots in the down kernel where its workgroups suffice, else with a row per pair); up to 512 tokens
with at most 8 rows per expert on average they walk the route's list in M-tiles of 32 rows. Cases sit on both sides of each line, at the smallest and largest sizes, with ids that are out of range
or name an expert twice, one expert taking every token, and glu segments stored scaled.
"""

from __future__ import annotations

import pytest
import torch

from helpers import assert_within_tolerance, form_of, oracle_fp64, packed_form, rand_case, to_device
from oracle import eager as O

pytestmark = pytest.mark.gpu


def _packed(c, device):
    from cernels_amd import ops

    d = to_device(c, device)
    layout = ops.LAYOUT_CONCAT if c["layout"] == "concat" else ops.LAYOUT_INTERLEAVED
    act = ops.ACT_SILU if c["act"] == "silu" else ops.ACT_GPTOSS
    pk = ops.pack_experts(d["W1"], d["W2"], layout=layout, act=act, gate_up_bias=d["b1"], down_bias=d["b2"])
    return ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], d["idx"].shape[1]).cpu()


SILU, GPT = ("concat", "silu", False), ("interleaved", "gptoss", True)
CASES = [
    # T, H, F, E, K, (layout, act, bias), ids, the form that the call takes
    (1, 64, 64, 1, 1, SILU, "plain", "few_sum"),  # one stage per projection: three of the four waves have none
    (1, 192, 320, 1024, 16, SILU, "plain", "few_rows"),  # 16 pairs in one token, partial last bundles
    (1, 2048, 192, 20, 16, SILU, "plain", "few_sum"),  # long rows of the result: the sum is in the down kernel
    (2, 2048, 2112, 3, 3, GPT, "twice", "few_sum"),  # 33 stages: eight shares of an expert, 5 + 7 x 4
    (3, 2048, 1088, 4, 3, SILU, "plain", "few_sum"),  # 17 stages: four shares
    (1, 1024, 512, 20, 16, SILU, "plain", "few_sum"),  # shorter ones with up to 8 H columns of glu over all experts
    (1, 1024, 576, 20, 16, SILU, "plain", "few_rows"),  # more
    (1, 192, 256, 40, 16, GPT, "plain", "few_sum"),  # or up to 5000
    (8, 64, 1088, 2, 2, GPT, "plain", "few_sum"),  # or two experts
    (16, 128, 192, 3, 1, GPT, "plain", "few_sum"),  # 16 pairs, the fused down's last
    (17, 128, 192, 3, 1, GPT, "plain", "few_rows"),  # 17: rows and combine
    (4, 576, 64, 9, 4, GPT, "twice", "few_sum"),
    (5, 320, 128, 6, 3, SILU, "twice", "few_sum"),  # an expert named twice by one token
    (11, 320, 128, 6, 3, SILU, "twice", "few_rows"),
    (7, 128, 64, 12, 2, SILU, "invalid", "few_sum"),
    (3, 128, 64, 4, 2, GPT, "none", "few_sum"),  # no valid id at all: zeros
    (20, 128, 64, 4, 2, SILU, "none", "few_rows"),
    (32, 128, 64, 512, 16, SILU, "plain", "few_rows"),  # 512 pairs, 2^20 ids read by the first projection's workgroups
    (32, 128, 128, 512, 16, SILU, "plain", "tiles"),  # more ids: tiles, with few tokens
    (32, 128, 576, 32, 16, GPT, "twice", "few_rows"),  # more than 8 rows per expert: 600000 ids
    (32, 128, 640, 32, 16, GPT, "twice", "grouped"),  # above
    (32, 128, 128, 512, 17, SILU, "plain", "tiles"),  # 544: the route's list (tiles)
    (32, 1088, 448, 64, 8, GPT, "same", "few_rows"),  # every token on the same experts
    (33, 128, 192, 64, 4, SILU, "invalid", "tiles"),  # 33 tokens: tiles
    (64, 256, 128, 32, 4, GPT, "plain", "tiles"),  # 8 rows per expert: tiles' last
    (65, 256, 128, 32, 4, GPT, "plain", "grouped"),  # above: the grouped GEMMs
    (512, 128, 64, 64, 1, SILU, "same", "tiles"),  # one expert with 512 rows: 16 tiles
    (513, 128, 64, 65, 1, SILU, "plain", "grouped"),
    (90, 192, 64, 40, 3, SILU, "twice", "tiles"),
]


def _case(T, H, Fi, E, K, kind, ids):
    layout, act, bias = kind
    c = rand_case(7 * T + K, T, H, Fi, E, K, layout=layout, act=act, bias=bias, std=0.05,
                  invalid=max(3, T // 4) if ids == "invalid" else 0)
    if ids == "twice":
        c["idx"][::2, K - 1] = c["idx"][::2, 0]
    elif ids == "same":
        c["idx"][:] = c["idx"][:1]
    elif ids == "none":
        c["idx"][:] = E + 5
    return c


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"T{c[0]}H{c[1]}F{c[2]}E{c[3]}k{c[4]}{c[5][1]}-{c[6]}")
def test_few_rows(device, case):
    c = _case(*case[:7])
    assert form_of(c) == case[7]
    print(f"[few rows {case}]", flush=True)
    out = _packed(c, device)
    ref = oracle_fp64(c)
    if case[6] == "none":
        assert not out.float().any()
    assert_within_tolerance(out, ref, str(case))


@pytest.mark.parametrize("gain", [3000.0, 1e-4, 2.0 ** -57])
@pytest.mark.parametrize("T,E,bias,form", [(5, 8, True, "few_sum"), (30, 8, True, "few_rows"), (40, 32, False, "tiles")],
                         ids=["fused", "rows", "tiles"])
def test_few_rows_scaled_segments(device, T, E, bias, form, gain):
    """Rows whose glu leaves fp16's range (or falls to its subnormals) are stored scaled; each row group meets the bar on its
    own scale, with columns 0-15 of two experts at zero so that scaled rows hold all-zero segments too. At 2^-57 glu lies near
    2^-115: the product of the row's, the fragment's and the routing weight's powers is subnormal, the results are not."""
    K = 3
    c = rand_case(T, T, 256, 192, E, K, std=0.05, bias=bias and gain > 1)
    assert form_of(c) == form
    for e in (0, 3):
        c["W1"][e, :16] = 0
    odd = torch.arange(1, T, 4)
    x = c["x"].float()
    x[odd] *= gain
    c["x"] = x.bfloat16()
    print(f"[few rows scaled T{T} gain {gain}]", flush=True)
    out = _packed(c, device)
    assert torch.isfinite(out.float()).all()
    ref = oracle_fp64(c)
    rest = torch.ones(T, dtype=torch.bool)
    rest[odd] = False
    assert_within_tolerance(out[odd], ref[odd], "scaled rows")
    assert_within_tolerance(out[rest], ref[rest], "other rows")


@pytest.mark.parametrize("T,form", [(4, "few_sum"), (24, "few_rows"), (60, "tiles")], ids=["fused", "rows", "tiles"])
def test_few_rows_nan_token(device, T, form):
    """A token with a nan gives an all-nan row; the others, which share its experts' workgroups, stay within the bar."""
    c = rand_case(T + 1, T, 128, 192, 10 if T == 4 else 32, 4)
    assert form_of(c) == form
    bad = T // 2
    c["x"][bad, 3] = float("nan")
    print(f"[few rows nan T{T}]", flush=True)
    out = _packed(c, device)
    keep = torch.tensor([t for t in range(T) if t != bad])
    assert torch.isnan(out[bad].float()).all()
    assert_within_tolerance(out[keep], oracle_fp64(c, keep), "nan token")


@pytest.mark.parametrize("T,E,act_id,form", [(1, 8, 0, "few_sum"), (30, 8, 1, "few_rows"), (40, 16, 2, "tiles"), (40, 16, 0, "tiles")])
def test_few_rows_nongated(device, T, E, act_id, form):
    from cernels_amd import ops

    g = torch.Generator().manual_seed(T + act_id)
    H, Fi, K = 192, 320, 2
    assert packed_form(T, H, Fi, E, K, act_id) == form
    x = torch.randn(T, H, generator=g).bfloat16()
    x[T // 2] *= 1000.0  # its segments are stored scaled
    w1 = (torch.randn(E, H, Fi, generator=g) * 0.05).bfloat16()
    w2 = (torch.randn(E, Fi, H, generator=g) * 0.05).bfloat16()
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).int()
    wt = torch.rand(T, K, generator=g)
    print(f"[few rows nongated T{T} act{act_id}]", flush=True)
    out = ops.megablocks_moe(*[t.contiguous().to(device) for t in (x, w1, w2, idx, wt)], K, act_id).cpu()
    ref = O.megablocks_fp64(x, idx, wt, w1, w2, act_id)
    big = torch.zeros(T, dtype=torch.bool)
    big[T // 2] = True
    assert_within_tolerance(out[big], ref[big], "scaled row")
    if T > 1:
        assert_within_tolerance(out[~big], ref[~big], "other rows")


@pytest.mark.parametrize("T,form", [(2, "few_sum"), (24, "few_rows"), (60, "tiles")], ids=["fused", "rows", "tiles"])
def test_few_rows_graph_replays(device, T, form):
    """Captured and replayed with new inputs in the same buffers, each replay equals the eager call bit for bit (nothing is
    kept between calls)."""
    from cernels_amd import ops

    c = rand_case(T + 2, T, 256, 192, 32, 4)
    assert form_of(c) == form
    d = to_device(c, device)
    pk = ops.pack_experts(d["W1"], d["W2"])
    out = torch.empty_like(d["x"])
    print(f"[few rows graph T{T}]", flush=True)
    ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], 4, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], 4, out=out)
    for i in range(3):
        n = to_device(rand_case(100 * i + T, T, 256, 192, 32, 4), device)
        d["x"].copy_(n["x"])
        d["idx"].copy_(n["idx"])
        d["w"].copy_(n["w"])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], 4))


@pytest.mark.parametrize("T,K,part,H,Fi,E,form", [(4, 4, 1, 2048, 832, 10, "few_sum"), (5, 3, 1, 2048, 2112, 6, "few_sum"),
                                                  (24, 4, 6, 192, 832, 32, "few_rows"), (64, 4, 40, 192, 832, 32, "tiles")],
                         ids=["fused", "fused-k3", "rows", "tiles"])
def test_few_rows_do_not_depend_on_the_other_tokens(device, T, K, part, H, Fi, E, form):
    """A token's row is the same bit for bit whether the call holds the other tokens or not (both calls of one form), some of
    which are stored scaled, and however the experts are numbered: its slots are summed in their own order, each from a
    reduction that is cut at places that only the layer's sizes fix. F gives 13 or 33 stages, which no number of shares divides."""
    from cernels_amd import ops

    c = rand_case(T + K, T, H, Fi, E, K, layout="interleaved", act="gptoss", bias=True, std=0.05)
    assert form_of(c) == packed_form(part, H, Fi, E, K, "gptoss") == form
    # two slots cancel exactly (equal experts, weights 1 and -1) beside small ones: what is left of a sum that was cut or ordered
    # otherwise shows in bf16
    for name in ("W1", "W2", "b1", "b2"):
        c[name][1] = c[name][0]
    c["idx"][:, 0], c["idx"][:, 1] = 0, 1
    c["w"] = torch.cat([torch.ones(T, 1), -torch.ones(T, 1), torch.rand(T, K - 2) * 2.0 ** -12], dim=1).bfloat16()
    c["idx"][0, K - 1] = 0  # an expert named twice
    c["x"][T - 1] = (c["x"][T - 1].float() * 3000.0).bfloat16()
    d = to_device(c, device)
    kw = dict(layout=ops.LAYOUT_INTERLEAVED, act=ops.ACT_GPTOSS)
    pk = ops.pack_experts(d["W1"], d["W2"], gate_up_bias=d["b1"], down_bias=d["b2"], **kw)
    print(f"[few rows neighbours T{T} K{K}]", flush=True)
    whole = ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], K)
    for t in range(0, T - part + 1, part):
        r = slice(t, t + part)
        some = ops.moe_experts_packed(d["x"][r].contiguous(), pk, d["idx"][r].contiguous(), d["w"][r].contiguous(), K)
        assert torch.equal(some, whole[r]), f"tokens {t}..{t + part - 1}"
    perm = torch.randperm(E, generator=torch.Generator().manual_seed(1)).to(device)  # expert e moves to place perm[e]
    inv = torch.argsort(perm)
    pk2 = ops.pack_experts(d["W1"][inv].contiguous(), d["W2"][inv].contiguous(), gate_up_bias=d["b1"][inv].contiguous(),
                           down_bias=d["b2"][inv].contiguous(), **kw)
    assert torch.equal(ops.moe_experts_packed(d["x"], pk2, perm[d["idx"].long()].int(), d["w"], K), whole)
