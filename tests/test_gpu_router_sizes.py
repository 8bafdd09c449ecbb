"""Router sizes at the edges of its kernels' tiles (16 tokens x 16 experts split over waves, 32 tokens on a stage ring, 128 x 64 tiled), with and
without the shared-expert gate's row: the bounds of test_gpu_router.py against the CPU oracle."""

from __future__ import annotations

import pytest
import torch

from oracle import eager as O
from test_gpu_router import _case, _ulp

pytestmark = pytest.mark.gpu

CASES = [
    # T, H, E, K, mode, S, bias
    (1, 16, 1, 1, O.ROUTER_SOFTMAX_TOPK, 0, False),     # no whole k-step of 32: only the half one
    (16, 48, 16, 3, O.ROUTER_TOPK_SOFTMAX, 0, True),
    (17, 2896, 17, 4, O.ROUTER_TOPK_SOFTMAX, 0, True),  # 90.5 k-steps over 16 waves
    (15, 1024, 16, 2, O.ROUTER_SOFTMAX_TOPK, 1, False),  # 17 rows with the gate
    (33, 528, 32, 5, O.ROUTER_SOFTMAX_TOPK, 2, True),    # 33 rows
    (40, 320, 63, 6, O.ROUTER_SOFTMAX_TOPK, 1, False),   # 64 rows: the largest fused
    (31, 176, 64, 6, O.ROUTER_SOFTMAX_TOPK, 1, False),   # 65 rows: logits, then selection
    (4096, 2064, 17, 3, O.ROUTER_TOPK_SOFTMAX, 0, True),  # 16 tokens per workgroup: the last of this width
    (4097, 2064, 17, 3, O.ROUTER_TOPK_SOFTMAX, 0, True),  # the stage ring: one token in the last workgroup, a quarter stage
    (4130, 2048, 32, 4, O.ROUTER_SOFTMAX_TOPK, 1, True),  # 33 rows with the gate
    (8193, 1040, 31, 4, O.ROUTER_SOFTMAX_TOPK, 1, False),  # 32 rows with the gate
    (8223, 2080, 9, 2, O.ROUTER_TOPK_SOFTMAX, 0, False),
    (8200, 1552, 64, 6, O.ROUTER_SOFTMAX_TOPK, 0, True),
    (256, 2048, 127, 8, O.ROUTER_SOFTMAX_TOPK, 1, True),  # the split kernel's last
    (257, 2048, 127, 8, O.ROUTER_SOFTMAX_TOPK, 1, True),  # the tiled kernel's first
    (1000, 592, 513, 10, O.ROUTER_TOPK_SOFTMAX, 0, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"T{c[0]}H{c[1]}E{c[2]}S{c[5]}")
def test_router_sizes(device, case):
    from cernels_amd import ops

    T, H, E, K, mode, S, bias = case
    x, w, b = _case(T + E, T, H, E + (S > 0), bias)
    print(f"[router sizes {case}]", flush=True)
    idx, wts, logits = (t.cpu() for t in ops.moe_router(x.to(device), w.to(device), None if b is None else b.to(device), K,
                                                        mode, want_logits=True, shared_slots=S))
    ref = O.router_logits(x, w, b)
    tol = _ulp(ref).double() + H * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((logits.float() - ref.float()).abs().double() <= tol).all())
    ridx, rw = O.router_select(logits[:, :E], K, mode)
    assert torch.equal(idx[:, :K].long(), ridx)
    assert bool(((wts[:, :K] - rw.float()).abs() <= _ulp(rw)).all())
    if S:
        assert torch.equal(idx[:, K:].long(), torch.arange(E, E + S).expand(T, S))
        sg = torch.sigmoid(logits[:, E:].double())
        assert bool(((wts[:, K:].double() - sg).abs() <= _ulp(sg)).all())
