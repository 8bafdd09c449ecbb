"""Packed experts on workgroup-sized items (128 rows x 8 weight fragments), against the fp64 oracle.

The ids give chosen experts run lengths around each edge of the rows (a 32-row block, a whole item, several), the other
experts the rest; odd numbers of 64-column groups and fragment counts that no item width divides; unselected experts and
invalid ids; an item's rows in one segment scale or several; both gated activations with and without bias, and non-gated.
"""

from __future__ import annotations

import pytest
import torch

from helpers import assert_within_tolerance, form_of, oracle_fp64, packed_form, rand_case, to_device
from oracle import eager as O

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 31, 32, 33, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 191, 192, 193, 255, 256, 257, 383, 384, 385]
# E, rows per expert on average, H, F: one for each line of the rule that chooses these items
FEW_ROWS, MANY_ROWS = (512, 40, 192, 320), (40, 300, 1088, 576)


def _ids(E, mean, seed):
    """Ids: expert e < len(EDGES) exactly EDGES[e] times, the others evenly up to the average."""
    rest = E * mean - sum(EDGES)
    n = E - len(EDGES)
    counts = EDGES + [rest // n + (i < rest % n) for i in range(n)]
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    return ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(seed))]


def _packed(c, device):
    from cernels_amd import ops

    d = to_device(c, device)
    layout = ops.LAYOUT_CONCAT if c["layout"] == "concat" else ops.LAYOUT_INTERLEAVED
    act = ops.ACT_SILU if c["act"] == "silu" else ops.ACT_GPTOSS
    pk = ops.pack_experts(d["W1"], d["W2"], layout=layout, act=act, gate_up_bias=d["b1"], down_bias=d["b2"])
    return ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], d["idx"].shape[1]).cpu()


def _case(shape, kind, seed=3, K=1):
    E, mean, H, Fi = shape
    layout, act, bias = kind
    ids = _ids(E, mean, seed)
    T = len(ids) // K
    c = rand_case(seed, T, H, Fi, E, K, layout=layout, act=act, bias=bias, std=0.05)
    c["idx"] = ids.reshape(T, K)  # a token may name an expert twice
    c["w"] = torch.rand(T, K, generator=torch.Generator().manual_seed(seed)).bfloat16()
    assert form_of(c) == "items"
    return c


@pytest.mark.parametrize("kind", [("concat", "silu", False), ("interleaved", "gptoss", True), ("concat", "silu", True)],
                         ids=["silu", "gptoss", "silu-bias"])
@pytest.mark.parametrize("shape", [FEW_ROWS, (520, 12, 64, 64), MANY_ROWS, (40, 300, 1344, 448)], ids=lambda s: "E%d-%drows-H%d-F%d" % s)
def test_items_row_edges(device, shape, kind):
    c = _case(shape, kind)
    print(f"[items {shape} {kind}]", flush=True)
    assert_within_tolerance(_packed(c, device), oracle_fp64(c), f"{shape} {kind}")


@pytest.mark.parametrize("K", [2, 5])
@pytest.mark.parametrize("shape", [FEW_ROWS, MANY_ROWS], ids=["few", "many"])
def test_items_several_slots(device, shape, K):
    """Several pairs per token: a row's token is not its pair, and the combine sums the slots."""
    c = _case(shape, ("interleaved", "gptoss", True), seed=7, K=K)
    print(f"[items {shape} K{K}]", flush=True)
    assert_within_tolerance(_packed(c, device), oracle_fp64(c), f"{shape} K{K}")


@pytest.mark.parametrize("shape", [FEW_ROWS, MANY_ROWS], ids=["few", "many"])
def test_items_scaled_nan_and_invalid(device, shape):
    """Every 50th token large enough that its glu is stored scaled, with all-zero segments in two experts; one token with a
    nan; some ids invalid (zero rows). Each group of rows meets the bar on its own scale."""
    c = _case(shape, ("concat", "silu", False), seed=5)
    T = c["x"].shape[0]
    for e in (16, 30):
        c["W1"][e, :16] = 0
    big = torch.zeros(T, dtype=torch.bool)
    big[::50] = True
    x = c["x"].float()
    x[big] *= 3000.0
    c["x"] = x.bfloat16()
    bad = 7
    c["x"][bad, 3] = float("nan")
    c["idx"][bad, 0] = 35
    none = torch.zeros(T, dtype=torch.bool)
    none[11::97] = True
    c["idx"][none, 0] = shape[0] + 2
    print(f"[items scaled {shape}]", flush=True)
    out = _packed(c, device)
    ref = oracle_fp64(c)
    assert torch.isnan(out[bad].float()).all()
    assert not out[none].float().any()
    rest = ~big & ~none
    rest[bad] = False
    assert_within_tolerance(out[big & ~none], ref[big & ~none], "scaled rows")
    assert_within_tolerance(out[rest], ref[rest], "other rows")


@pytest.mark.parametrize("act_id", [0, 1, 2])
@pytest.mark.parametrize("shape", [(512, 40, 192, 320), (40, 300, 1088, 1088)], ids=["few", "many"])
def test_items_nongated(device, shape, act_id):
    from cernels_amd import ops

    E, mean, H, Fi = shape
    g = torch.Generator().manual_seed(act_id)
    idx = _ids(E, mean, act_id)[:, None].int()
    assert packed_form(len(idx), H, Fi, E, 1, act_id) == "items"
    x = torch.randn(len(idx), H, generator=g).bfloat16()
    w1 = (torch.randn(E, H, Fi, generator=g) * 0.05).bfloat16()
    w2 = (torch.randn(E, Fi, H, generator=g) * 0.05).bfloat16()
    wt = torch.rand(len(idx), 1, generator=g)
    print(f"[items nongated {shape} act{act_id}]", flush=True)
    out = ops.megablocks_moe(*[t.contiguous().to(device) for t in (x, w1, w2, idx, wt)], 1, act_id).cpu()
    assert_within_tolerance(out, O.megablocks_fp64(x, idx, wt, w1, w2, act_id), f"{shape} act{act_id}")
