"""GPU parity of both forms of the split merge of ``sparse_attention`` (a workgroup per
(row, head) for few of them, eight rows a workgroup for more) against the CPU oracle,
on both sides of the line between them and at every remainder of four splits.

Bar: fp32 scores over up to 128 dims, sums over at most 64 keys, as in one part; the
merge adds one rounded product per split: 2^-24 (sqrt(128 + 64) + 17) = 2e-6 of the
oracle's norm."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from linattn_amd.kernels.block_sparse import sparse_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hkv,G,Tq,splits", [
    (1, 1, 1, 1, 2),
    (3, 2, 4, 1, 16),        # a decode step
    (1, 2, 4, 256, 3),       # 2048 (row, head)s: the last of the few
    (1, 1, 1, 2049, 5),      # one more: the last workgroup holds one row
    (2, 2, 2, 515, 2),
    (1, 2, 1, 1030, 17),
])
def test_merge_matches_oracle(dev, D, B, Hkv, G, Tq, splits):
    g = torch.Generator().manual_seed(splits)
    q = torch.randn(B, Hkv * G, Tq, D, generator=g)
    k = torch.randn(B, Hkv, 300, D, generator=g)
    v = torch.randn(B, Hkv, 300, D, generator=g)
    ids = torch.rand(B, Hkv, Tq, 100, generator=g).argsort(-1)[..., :32].to(torch.int32)
    ids[:, :, ::3, ::2] = -1  # parts without a key, and rows without any
    ids[:, :, 1::5] = -1
    got = sparse_attention(q.to(dev), k.to(dev), v.to(dev), ids.to(dev), unit=2, num_splits=splits)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=2)
    got = got.cpu().double().numpy()
    assert np.linalg.norm(got - want) < 2e-6 * np.linalg.norm(want) + 1e-30
    assert (got[:, :, 1::5] == 0).all()
    wide = torch.full((B, Hkv * G, Tq, D + 3), 7.0, dtype=torch.bfloat16, device=dev)
    sparse_attention(q.to(dev), k.to(dev), v.to(dev), ids.to(dev), unit=2, num_splits=splits,
                     out=wide[..., 1:D + 1])  # rows off a 4-byte boundary, neighbours kept
    assert (wide[..., :1] == 7).all() and (wide[..., D + 1:] == 7).all()
    assert np.linalg.norm(wide[..., 1:D + 1].cpu().double().numpy() - want) < 3e-3 * np.linalg.norm(want) + 1e-30
