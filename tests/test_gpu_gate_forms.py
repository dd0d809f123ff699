"""GPU parity of the block gates in every form their scores are computed in
(decode rows, rows of q as stored, tiles; csrc/block_select.hip) against the CPU
oracle: lists bit for bit, at the edges of each form's rows and columns."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from linattn_amd.kernels.prefill import block_select_hip
from linattn_amd.kernels.routing import gate_select_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,Tq,nkb,D,dtype", [
    (8, 2, 1, 1, 128, torch.bfloat16),     # decode form: one column, its most rows
    (8, 2, 2, 65, 128, torch.float32),
    (4, 4, 8, 64, 64, torch.float16),
    (4, 4, 9, 33, 64, torch.float16),      # one row more than the decode form takes
    (32, 2, 1, 65, 128, torch.bfloat16),   # 4-row tiles: groups the decode form has no room for
    (16, 2, 4, 64, 128, torch.float32),
    (16, 2, 5, 64, 128, torch.float32),    # one row more than those take
    (4, 4, 1, 63, 192, torch.bfloat16),    # dims it has no room for
    (4, 2, 3, 66, 33, torch.float16),
    (8, 2, 15, 31, 64, torch.bfloat16),    # tiles: too few rows
    (4, 2, 16, 33, 128, torch.bfloat16),   # rows: the fewest, a column past a group
    (2, 1, 64, 32, 72, torch.bfloat16),
    (2, 1, 65, 40, 128, torch.float32),
    (2, 1, 129, 8, 8, torch.float16),
    (2, 1, 130, 100, 128, torch.bfloat16),
    (2, 1, 40, 20, 136, torch.bfloat16),   # more dims than the row form holds
    (2, 1, 40, 20, 60, torch.bfloat16),    # dims not in whole pieces
])
def test_gates_bit_exact_in_every_form(dev, hq, hkv, Tq, nkb, D, dtype):
    g = torch.Generator().manual_seed(11)
    bs = 4
    T = nkb * bs - 1
    q = torch.randn(2, hq, Tq, D, generator=g).to(dtype)
    k = torch.randn(2, hkv, T, D, generator=g).to(dtype)
    for off in sorted({0, max(0, T - Tq)}):
        ids, counts = gate_select_hip(q.to(dev), k.to(dev), block=bs, topk=5, offset=off)
        ref = oracle.gate_select(q.float(), k.float(), block=bs, topk=5, offset=off)
        assert np.array_equal(ids.cpu().numpy(), ref)
        assert np.array_equal(counts.cpu().numpy(), (ref >= 0).sum(-1))
    # rows of a wider tensor (their pieces start off a 16-byte boundary)
    wide = torch.zeros(2, hq, Tq, D + 4, dtype=dtype)
    wide[..., 2:-2] = q
    ids2, _ = gate_select_hip(wide.to(dev)[..., 2:-2], k.to(dev), block=bs, topk=5, offset=off)
    assert torch.equal(ids2, ids)


def test_gates_tie_to_the_lowest_block(dev):
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 2, 70, 64, generator=g)
    q[:, :, :35] = 0.0
    q[:, :, 20:25] = -0.0
    k = torch.randn(1, 1, 300, 64, generator=g)
    ids, _ = gate_select_hip(q.to(dev), k.to(dev), block=8, topk=6, offset=230)
    assert np.array_equal(ids.cpu().numpy(), oracle.gate_select(q, k, block=8, topk=6, offset=230))


@pytest.mark.parametrize("T,topk,sink,window", [(64, 1, 0, 0), (200, 3, 2, 1), (1000, 16, 1, 4),
                                                (4200, 16, 1, 4), (4200, 70, 70, 3)])
def test_block_lists_place_sinks_and_windows(dev, T, topk, sink, window):
    g = torch.Generator().manual_seed(T)
    q = torch.randn(1, 4, T, 64, generator=g).bfloat16()
    k = torch.randn(1, 2, T, 64, generator=g).bfloat16()
    ids, counts = block_select_hip(q.to(dev), k.to(dev), topk=topk, sink_blocks=sink,
                                   window_blocks=window)
    ref = oracle.block_select(q, k, block=64, topk=topk, sink_blocks=sink, window_blocks=window)
    ref = ref[0] if isinstance(ref, tuple) else ref
    n = min(ref.shape[-1], ids.shape[-1])
    assert np.array_equal(ids.cpu().numpy()[..., :n], ref[..., :n])
    assert np.array_equal(counts.cpu().numpy(), (ref >= 0).sum(-1))


@pytest.mark.parametrize("nb,D", [(1, 2), (63, 30), (64, 32), (65, 34), (130, 66), (66, 33), (70, 160)])
def test_pooled_scores_in_every_tile_form(dev, nb, D):
    """Pooled q on 64 x 64 tiles: partial tiles and slices of 32 dims, staged in
    pairs of dims (even D) or one by one (odd D)."""
    g = torch.Generator().manual_seed(D)
    q = torch.randn(2, 4, 4 * nb - 1, D, generator=g).bfloat16()
    k = torch.randn(2, 2, 4 * nb - 1, D, generator=g).bfloat16()
    ids, counts = block_select_hip(q.to(dev), k.to(dev), block=4, topk=7, sink_blocks=1, window_blocks=1)
    ref = oracle.block_select(q, k, block=4, topk=7, sink_blocks=1, window_blocks=1)
    ref = ref[0] if isinstance(ref, tuple) else ref
    n = min(ref.shape[-1], ids.shape[-1])
    assert np.array_equal(ids.cpu().numpy()[..., :n], ref[..., :n])
    assert np.array_equal(counts.cpu().numpy(), (ref >= 0).sum(-1))
