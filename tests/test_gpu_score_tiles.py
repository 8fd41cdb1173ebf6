"""The tile score kernel (D = 128) against the oracle: every head count it is
built for, page counts around its 64-page tile, ragged launches on both sides
of the size from which a block waits for its group's length, and operands that
go to the general kernel.  Scores are sums in a fixed order: the same bits."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from helpers import randn, to_bits

pytestmark = pytest.mark.gpu

D = 128


def _operands(G, R, P, dtype, seed, dev):
    a, b = (randn((G, P, D), dtype, seed=seed + i) for i in range(2))
    lo, hi = torch.minimum(a, b), torch.maximum(a, b)
    q = randn((G, R, D), "f32", seed=seed + 2)
    q[:, :, ::7] = 0.0          # zeros of both signs take the minimum
    q[:, :, 3] = -0.0
    q[0, 0, 5] = float("inf")
    return q.to(dev), lo.to(dev), hi.to(dev)


def _want(q, lo, hi, dtype):
    return oracle.quest_score(q.cpu().numpy(), to_bits(lo), to_bits(hi), dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_scores_every_head_count(dev, dtype, R):
    from headinfer import kernels

    for G, P in ((1, 1), (3, 63), (2, 64), (3, 65), (1, 300)):
        q, lo, hi = _operands(G, R, P, dtype, 10 * R + P, dev)
        got = kernels.fused_quest_score(q, lo, hi)
        want = _want(q, lo, hi, dtype)
        assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32)), (G, P)


def test_scores_off_the_16_byte_grid(dev):
    """Metadata that starts two bytes into a row of 16 goes to the general kernel: the same scores."""
    from headinfer import kernels

    q, lo, hi = _operands(2, 5, 130, "bf16", 7, dev)
    odd = [torch.empty(t.numel() + 2, dtype=t.dtype, device=dev)[2:].view(t.shape).copy_(t) for t in (lo, hi)]
    assert odd[0].data_ptr() % 16
    a, b = kernels.fused_quest_score(q, *odd), kernels.fused_quest_score(q, lo, hi)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def test_queries_off_the_16_byte_grid(dev):
    """Queries that start four bytes into a row of 16: the scalar loads need no more than a word's alignment."""
    from headinfer import kernels

    for R in (1, 4, 7, 8):
        q, lo, hi = _operands(3, R, 130, "bf16", 11, dev)
        odd = torch.empty(q.numel() + 1, dtype=q.dtype, device=dev)[1:].view(q.shape).copy_(q)
        assert odd.data_ptr() % 16 == 4
        got = kernels.fused_quest_score(odd, lo, hi)
        assert np.array_equal(got.cpu().numpy().view(np.uint32), _want(q, lo, hi, "bf16").view(np.uint32)), R


@pytest.mark.parametrize("R", [4, 7, 8])  # (8: some queries outside the scalar registers)
@pytest.mark.parametrize("G,P", [(4, 200), (9, 1900)])  # 16 and 270 blocks
def test_ragged_scores_select_the_same_pages(dev, G, P, R):
    from headinfer import kernels

    sink, recent, bs, k = 64, 256, 16, 20
    q, lo, hi = _operands(G, R, P, "bf16", 5, dev)
    q[0, 0, 5] = 1.0
    pages = [int(x) for x in np.linspace(0, P, G)]
    pages[1] = 65
    lengths = torch.tensor([sink + p * bs + recent - 1 for p in pages], dtype=torch.int32, device=dev)
    sel = torch.empty((G, R, k), dtype=torch.int32, device=dev)
    plan = torch.empty((G, min(P, R * k)), dtype=torch.int32, device=dev)
    masks = torch.empty(plan.shape, dtype=torch.uint8, device=dev)
    counts = torch.empty((G,), dtype=torch.int32, device=dev)
    kernels.quest_select_ragged(q, lo, hi, lengths, k, sink=sink, recent=recent, block_size=bs, sel_pages=sel,
                                plan_pages=plan, plan_masks=masks, plan_counts=counts)
    for g, p in enumerate(pages):
        n = min(k, p)
        assert bool((sel[g, :, n:] == -1).all())
        if n:
            sc = _want(q[g:g + 1], lo[g:g + 1, :p], hi[g:g + 1, :p], "bf16")[0]
            assert np.array_equal(sel[g, :, :n].cpu().numpy(), oracle.topk_sorted(sc, n)), g
