"""Routing in a router's own types (int64 ids, bf16 weights): every native route reads them as the casts to int32 and fp32
would give them, so the output equals the cast call's bit for bit, on each path of the packed and decode entries."""

from __future__ import annotations

import pytest
import torch

from helpers import assert_within_tolerance, oracle_fp64, rand_case, to_device

pytestmark = pytest.mark.gpu

TYPES = [(torch.int64, torch.bfloat16), (torch.int64, torch.float32), (torch.int32, torch.bfloat16)]
CASES = [
    # T, H, F, E, K, ids
    (3, 128, 64, 8, 2, "plain"),       # packed: fused few tokens
    (9, 128, 64, 8, 3, "twice"),       # rows and combine, an expert named twice
    (40, 128, 64, 64, 3, "plain"),     # the route's list, 32-row tiles
    (341, 128, 64, 4, 3, "invalid"),   # grouped GEMMs; 1023 pairs, one short of a route tile
    (1025, 64, 64, 7, 1, "plain"),     # 1025 pairs: an odd last chunk of ids
    (5000, 64, 64, 1024, 6, "plain"),  # route of several launches
]


@pytest.mark.parametrize("types", TYPES, ids=["i64bf16", "i64f32", "i32bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"T{c[0]}E{c[3]}k{c[4]}{c[5]}")
def test_packed_pair_types(device, case, types):
    from cernels_amd import ops

    T, H, Fi, E, K, ids = case
    c = rand_case(T, T, H, Fi, E, K, invalid=9 if ids == "invalid" else 0)
    if ids == "twice":
        c["idx"][:, 2] = c["idx"][:, 0]
    d = to_device(c, device)
    pk = ops.pack_experts(d["W1"], d["W2"])
    idx, w = c["idx"].to(types[0]).to(device), c["w"].to(types[1]).to(device)
    if types[0] is torch.int64 and ids == "invalid":
        idx = torch.where(idx < 0, idx - 2**40, idx)  # the low 32 bits are the id
    print(f"[pair types packed {case} {types}]", flush=True)
    want = ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], K)
    got = ops.experts_packed(d["x"], pk, idx, w)
    assert torch.equal(got, want)
    assert_within_tolerance(got.cpu()[:64], oracle_fp64(c, slice(0, 64)), str(case))


@pytest.mark.parametrize("types", TYPES, ids=["i64bf16", "i64f32", "i32bf16"])
@pytest.mark.parametrize("T,K", [(1, 1), (1, 8), (7, 3), (32, 8), (64, 4)])
def test_decode_pair_types(device, T, K, types):
    from cernels_amd import ops

    c = rand_case(T + K, T, 256, 128, 24, K, invalid=T // 8)
    d = to_device(c, device)
    print(f"[pair types decode T{T} K{K} {types}]", flush=True)
    want = ops.moe_experts(d["x"], d["W1"], d["W2"], d["idx"], d["w"], K, decode=True)
    got = ops.experts_decode(d["x"], d["W1"], d["W2"], c["idx"].to(types[0]).to(device), c["w"].to(types[1]).to(device))
    assert torch.equal(got, want)


def test_loaders_refuse_what_they_refused(device):
    """The loaders' checks raise as the ops' do, whatever the routing's types; other types are cast."""
    from cernels_amd import ops
    from cernels_amd.configs.modules import Experts
    from cernels_amd.kops.registry import cohere2_moe_experts as c2

    c = rand_case(1, 12, 128, 64, 8, 2)
    d = to_device(c, device)
    m = Experts(d["W1"], d["W2"])
    idx, w = c["idx"].to(device), c["w"].to(device)
    for f in (c2.kernel, c2.decode_kernel):
        good = f(d["x"], idx, w, m)
        assert torch.equal(good, f(d["x"], idx.to(torch.int16), w.double(), m))
        assert torch.equal(good, f(d["x"].t().contiguous().t(), idx.t().contiguous().t(), w.t().contiguous().t(), m))
        for bad in ((d["x"].float(), idx, w), (d["x"].cpu(), idx, w), (d["x"], idx.cpu(), w), (d["x"], idx, w[:, :1]),
                    (d["x"][:, :64].contiguous(), idx, w), (d["x"][:5], idx, w)):
            with pytest.raises(RuntimeError):
                f(*bad, m)
    with pytest.raises(RuntimeError):
        ops.moe_experts(d["x"], d["W1"], d["W2"], idx, d["w"], 2, decode=True)  # the op itself keeps to int32
    with pytest.raises(RuntimeError):
        ops.moe_experts_packed(d["x"], ops.pack_experts(d["W1"], d["W2"]), idx, d["w"], 2)


@pytest.mark.parametrize("T,E,K", [(1, 1, 1), (16, 1, 1), (32, 512, 16), (33, 40, 4), (512, 1024, 16), (700, 520, 16), (300, 4, 3),
                                   (5000, 1024, 6)])
def test_packed_typed_stays_in_its_workspace(device, T, E, K):
    """Each form of the packed path, with ids and weights to convert, in a workspace of exactly the stated size (the smallest
    layer, where the parts that share space lie closest): the bytes behind it stay as they were, the result is the op's."""
    import ctypes

    from cernels_amd import _native, ops

    H = Fi = 64
    c = rand_case(T + K, T, H, Fi, E, K)
    d = to_device(c, device)
    pk = ops.pack_experts(d["W1"], d["W2"])
    idx, w = c["idx"].long().to(device), c["w"].bfloat16().to(device)
    L = _native.lib()
    n = L.cernels_moe_experts_workspace_bytes(T, H, Fi, E, K)
    ws = torch.full((n + 4096,), 0x5A, dtype=torch.uint8, device=device)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=device)
    print(f"[workspace T{T} E{E} K{K}]", flush=True)
    st = L.cernels_moe_experts_packed_typed(
        d["x"].data_ptr(), pk.gate_up.data_ptr(), None, pk.down.data_ptr(), None, idx.data_ptr(), _native.INDEX_I64, w.data_ptr(),
        _native.WEIGHT_BF16, T, H, Fi, E, K, 0, _native.ACT_SILU, out.data_ptr(), ws.data_ptr(), ctypes.c_size_t(n),
        torch.cuda.current_stream().cuda_stream)
    assert st == 0
    assert bool((ws[n:] == 0x5A).all())
    assert torch.equal(out, ops.moe_experts_packed(d["x"], pk, d["idx"], d["w"], K))
    assert_within_tolerance(out.cpu()[:64], oracle_fp64(c, slice(0, 64)), f"T{T} E{E} K{K}")
