"""GPU parity of the one-kernel per-head Quest selection
(``la_quest_select_heads``) with the CPU oracle, and with the two-launch path
(scores, then top-k) on forms both take: lists bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from linattn_amd.kernels.quest_pages import _topk, page_scores_hip, page_update_hip, quest_select_hip

pytestmark = pytest.mark.gpu


def _two_launches(q, mins, maxs, *, page_size, topk, offset):
    k = max(1, min(topk, mins.shape[2]))
    ids, counts, _ = _topk(page_scores_hip(q, mins, maxs), k=k, width=k, group=1, order=0,
                           pos_offset=offset, pos_unit=page_size, force_own=True)
    return ids, counts


@pytest.mark.parametrize("B,hq,hkv,Tq,pages,D,topk,dtype", [
    (1, 2, 2, 1, 1, 64, 4, torch.float32),
    (1, 8, 8, 1, 256, 64, 16, torch.float32),     # four waves a row
    (2, 4, 2, 3, 65, 72, 9, torch.bfloat16),      # two slots a lane
    (1, 4, 1, 40, 64, 128, 64, torch.bfloat16),   # every page kept
    (1, 4, 1, 40, 63, 128, 70, torch.float32),
    (1, 2, 1, 1500, 130, 64, 5, torch.bfloat16),  # many rows: one wave each
    (1, 8, 8, 5, 257, 128, 33, torch.float32),
    (2, 2, 2, 2, 512, 64, 200, torch.bfloat16),
    (1, 2, 2, 1, 1000, 200, 256, torch.float32),
    # both sides of where two launches take over: rows, k, dims, heads a KV head
    (1, 8, 8, 64, 257, 128, 9, torch.bfloat16),
    (1, 9, 9, 57, 257, 128, 9, torch.bfloat16),
    (1, 4, 4, 600, 300, 64, 64, torch.float32),
    (1, 4, 2, 5, 300, 64, 128, torch.float32),
    (1, 4, 2, 5, 300, 64, 129, torch.float32),
    (1, 2, 2, 3, 256, 128, 65, torch.bfloat16),
    (1, 2, 2, 1100, 256, 128, 65, torch.bfloat16),
])
def test_lists_match_oracle(dev, B, hq, hkv, Tq, pages, D, topk, dtype):
    ps = 4
    T = pages * ps - 1
    g = torch.Generator().manual_seed(pages)
    q = torch.randn(B, hq, Tq, D, generator=g).to(dtype)
    k = torch.randn(B, hkv, T, D, generator=g).to(dtype)
    q[:, :, 0, :5] = torch.tensor([0.0, -0.0, 1.0, -1.0, 0.0], dtype=dtype)
    mins, maxs = page_update_hip(k.to(dev), ps)
    omin, omax = oracle.page_bounds(k, ps)
    for off in sorted({0, max(0, T - Tq)}):
        ids, counts = quest_select_hip(q.to(dev), mins, maxs, page_size=ps, topk=topk, offset=off,
                                       gqa_union=False)
        ref = oracle.quest_select(q, omin, omax, page_size=ps, topk=topk, offset=off,
                                  gqa_union=False)
        assert np.array_equal(ids.cpu().numpy(), ref)
        assert np.array_equal(counts.cpu().numpy(), (ref >= 0).sum(-1))
        ids2, counts2 = _two_launches(q.to(dev), mins, maxs, page_size=ps, topk=topk, offset=off)
        assert torch.equal(ids, ids2) and torch.equal(counts, counts2)


def test_ties_and_special_values_rank_as_in_two_launches(dev):
    g = torch.Generator().manual_seed(0)
    q = torch.randn(1, 4, 6, 64, generator=g)
    k = torch.randn(1, 4, 300, 64, generator=g)
    k[:, :, 40:200] = k[:, :, 40:41]  # pages that tie
    q[0, 0, 0] = 0.0
    q[0, 1, 1, 3], q[0, 1, 2, 3], q[0, 2, 3, 1] = float("inf"), float("-inf"), float("nan")
    k[0, 3, 130, 2], k[0, 3, 250, 2] = float("inf"), float("-inf")
    mins, maxs = page_update_hip(k.to(dev), 4)
    got = quest_select_hip(q.to(dev), mins, maxs, page_size=4, topk=20, offset=280, gqa_union=False)
    want = _two_launches(q.to(dev), mins, maxs, page_size=4, topk=20, offset=280)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("page,topk", [(8, 12), (4, 200), (2, 256), (1, 256)])
def test_ragged_positions_equal_one_call_per_sequence(dev, page, topk):
    """(One kernel for every k and row count it has room for: the other form takes a
    call per sequence.)"""
    g = torch.Generator().manual_seed(1)
    q = torch.randn(3, 4, 1, 64, generator=g).to(dev)
    k = torch.randn(3, 4, 900, 64, generator=g).to(dev)
    mins, maxs = page_update_hip(k, page)
    pos = torch.tensor([0, 433, 899], dtype=torch.int32, device=dev)
    ids, counts = quest_select_hip(q, mins, maxs, page_size=page, topk=topk, gqa_union=False, positions=pos)
    for b in range(3):
        one, n = _two_launches(q[b:b + 1], mins[b:b + 1], maxs[b:b + 1], page_size=page, topk=topk,
                               offset=int(pos[b]))
        assert torch.equal(ids[b:b + 1], one) and torch.equal(counts[b:b + 1], n)
