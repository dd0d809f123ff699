"""GPU parity of the tiled form of ``sparse_attention`` (many queries with
lists of their own over a contiguous bf16 cache, csrc/list_tile.hip) against
the CPU oracle, at the edges of its tiles, masks and rules.

Bars: fp32 outputs within 2e-6 of the oracle's norm: scores are exact bf16
products summed in fp32 over 128 dims, weights fp32, sums over at most 1100
keys, about 2^-24 sqrt(128 + 1100) = 2e-6 at the worst; bf16 outputs 3e-3 (half
an ulp of 8 bits is 2^-9 = 2e-3).
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import oracle
from linattn_amd import _native as N
from linattn_amd.kernels import block_sparse
from linattn_amd.kernels.block_sparse import sparse_attention

pytestmark = pytest.mark.gpu


def _inputs(B, Hkv, G, Tq, T, seed=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hkv * G, Tq, 128, generator=g).bfloat16()
    k = torch.randn(B, Hkv, T, 128, generator=g).bfloat16()
    v = torch.randn(B, Hkv, T, 128, generator=g).bfloat16()
    return q, k, v


def _lists(B, L, rows, T, unit, share, seed=1):
    """Random lists of `share` of the units, an unreachable unit and a few -1 among them."""
    g = torch.Generator().manual_seed(seed)
    nu = -(-T // unit)
    n = max(1, int(nu * share))
    ids = torch.rand(B, L, rows, nu + 1, generator=g).argsort(-1)[..., :n].to(torch.int32)
    return torch.where(torch.rand(ids.shape, generator=g) < 0.05, -1, ids).contiguous()


def _run(dev, q, k, v, ids, *, tiled=True, counts=None, kv_len=None, **kw):
    """The call, checking that its workspace says tiles (the row form of these
    sizes needs none or split partials only)."""
    seen = []
    lib = N.load()
    orig = lib.la_sparse_attention_workspace

    def workspace(a, kv):
        n = orig(a, kv)
        a._obj.num_splits = 1 if a._obj.N <= 1024 else 2
        seen.append(n > orig(a, kv))
        a._obj.num_splits = kw.get("num_splits", 0)
        return n

    lib.la_sparse_attention_workspace = workspace
    try:
        out = sparse_attention(q.to(dev), k.to(dev), v.to(dev), ids.to(dev),
                               counts=None if counts is None else counts.to(dev),
                               kv_len=None if kv_len is None else kv_len.to(dev), **kw)
    finally:
        lib.la_sparse_attention_workspace = orig
    assert tiled is None or seen == [tiled]
    return out.cpu().double().numpy()


def _check(got, want, tol):
    assert np.isfinite(got).all()
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < tol, err
    # no row is off by itself: each within the bar of its own norm (rows of few keys are
    # long, and rounding is relative) and 4 times that of the average row (rows of many
    # keys are short: their terms cancel, their errors do not)
    rows, own = np.linalg.norm(got - want, axis=-1), np.linalg.norm(want, axis=-1)
    bar = tol * (own + 4 * np.linalg.norm(want) / np.sqrt(rows.size))
    assert (rows < bar).all(), (rows / bar).max()


@pytest.mark.parametrize("G,per_head,Tq,T,unit", [
    (1, False, 1025, 1000, 1),    # one query past a whole number of tiles
    (4, False, 1056, 1000, 1),    # exact tiles, a partial last key block
    (2, True, 511, 1024, 1),
    (8, False, 1030, 705, 64),
    (4, True, 257, 1088, 64),
    (3, True, 350, 1000, 64),     # group sizes without a tile of their own
    (4, True, 260, 1000, 128),    # units of two key blocks
    (4, True, 260, 1001, 16),
    (4, True, 260, 1001, 24),     # units that straddle key blocks
])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_tiles_match_oracle(dev, G, per_head, Tq, T, unit, out):
    B, Hkv = 2, 2
    q, k, v = _inputs(B, Hkv, G, Tq, T)
    ids = _lists(B, Hkv * G if per_head else Hkv, Tq, T, unit, 0.6)
    off = max(0, T - Tq)
    got = _run(dev, q, k, v, ids, unit=unit, causal=True, offset=off, out_dtype=out)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=unit, causal=True, offset=off)
    _check(got, want, 2e-6 if out == torch.float32 else 3e-3)


def test_tiles_ragged_counts_and_shared_lists(dev):
    q, k, v = _inputs(2, 2, 4, 300, 900)
    lens = torch.tensor([517, 900], dtype=torch.int32)
    for b in range(2):  # what lies past a sequence's length is never read
        k[b, :, int(lens[b]):] = float("nan")
        v[b, :, int(lens[b]):] = float("nan")
    ids = _lists(2, 8, 300, 900, 1, 0.7)
    g = torch.Generator().manual_seed(5)
    counts = torch.randint(0, ids.shape[-1] + 1, ids.shape[:3], generator=g).to(torch.int32)
    got = _run(dev, q, k, v, ids, unit=1, counts=counts, kv_len=lens, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=1, counts=counts.numpy(),
                               kv_len=lens.tolist())
    _check(got, want, 2e-6)
    # one list for every query, and lists expanded over batch and heads (stride 0)
    for ids1 in (_lists(2, 8, 1, 517, 1, 0.9), _lists(1, 1, 300, 517, 1, 0.9).expand(2, 8, -1, -1)):
        got = _run(dev, q, k, v, ids1, unit=1, causal=True, offset=300, kv_len=lens,
                   out_dtype=torch.float32)
        want = oracle.attend_lists(q, k, v, ids1.numpy(), unit=1, causal=True, offset=300,
                                   kv_len=lens.tolist())
        _check(got, want, 2e-6)


@pytest.mark.parametrize("unit", [1, 64])
def test_tiles_leave_units_listed_twice_to_the_rows(dev, unit):
    """A unit listed twice counts twice (block_sparse.py:62-68)."""
    q, k, v = _inputs(1, 2, 4, 300, 1000)
    ids = _lists(1, 8, 300, 1000, unit, 0.6)
    ids[:, :, 5::7, 0] = ids[:, :, 5::7, 1]
    got = _run(dev, q, k, v, ids, unit=unit, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=unit)
    _check(got, want, 2e-6)


@pytest.mark.parametrize("unit,per_head", [(1, True), (1, False), (64, True)])
def test_tiles_whose_every_row_lists_a_unit_twice(dev, unit, per_head):
    """Whole tiles (32 queries), all but one row of one, and one list for every query."""
    q, k, v = _inputs(1, 2, 4, 400, 1000)
    ids = _lists(1, 8 if per_head else 2, 400, 1000, unit, 0.6)
    ids[..., 1] = ids[..., 0] = 3
    ids[:, 1, 40, 1] = -1
    ids[:, :, 64:130, 1] = -1
    got = _run(dev, q, k, v, ids, unit=unit, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=unit)
    _check(got, want, 2e-6)
    one = ids[:, :, :1].contiguous()
    got = _run(dev, q, k, v, one, unit=unit, out_dtype=torch.float32)
    _check(got, oracle.attend_lists(q, k, v, one.numpy(), unit=unit), 2e-6)


@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_long_lists_left_to_the_rows_in_parts(dev, G):
    """More than 1024 entries: the row kernel takes a left row's list in parts; some
    rows' counts leave a part, or all of them, empty."""
    Tq = 130 * 8 // G + 3
    q, k, v = _inputs(1, 2, G, Tq, 2000)
    ids = _lists(1, 2, Tq, 2000, 1, 0.9)
    ids[:, :, ::2, 0] = ids[:, :, ::2, 1]
    g = torch.Generator().manual_seed(4)
    counts = torch.randint(2, ids.shape[-1] + 1, ids.shape[:3], generator=g).to(torch.int32)
    counts[:, :, 4:8] = torch.tensor([0, 1, 900, 1025], dtype=torch.int32)
    ids[:, :, :2] = -1
    got = _run(dev, q, k, v, ids, unit=1, counts=counts, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=1, counts=counts.numpy())
    _check(got, want, 2e-6)


def test_tiles_keep_unlisted_values_out(dev):
    """Infinities, NaN and huge values reach only the rows that list them."""
    q, k, v = _inputs(1, 2, 4, 300, 1000)
    ids = _lists(1, 8, 300, 1000, 1, 0.6)
    ids[ids == 130] = -1
    ids[ids == 500] = -1
    clean = _run(dev, q, k, v, ids, unit=1, out_dtype=torch.float32)
    v[0, 0, 130, 3], k[0, 1, 500, 7], k[0, 0, 130, 9] = float("inf"), float("nan"), 3e38
    got = _run(dev, q, k, v, ids, unit=1, out_dtype=torch.float32)
    _check(got, clean, 2e-6)
    q[0, 3, 17] = float("nan")  # one query's values stay its own
    got = _run(dev, q, k, v, ids, unit=1, out_dtype=torch.float32)
    assert np.isnan(got[0, 3, 17]).all() or (got[0, 3, 17] == 0).all()
    got[0, 3, 17] = clean[0, 3, 17]
    _check(got, clean, 2e-6)


def test_tiles_that_share_little_go_to_the_rows(dev):
    """Lists so short that a tile's union is many times any of them."""
    q, k, v = _inputs(1, 2, 4, 1100, 16000)
    ids = _lists(1, 8, 1100, 16000, 64, 5.1 / 250)
    ids[:, :, 512:, 0] = 7  # (and ones whose rows share a block)
    ids[:, :, 512:, 1:] = -1
    got = _run(dev, q, k, v, ids, unit=64, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=64)
    _check(got, want, 2e-6)


@pytest.mark.parametrize("unit,per_head,given", [(8, False, "counts"), (8, True, "pad"),
                                                 (64, True, "counts"), (1, False, "counts")])
def test_wide_lists_decide_by_what_they_hold(dev, unit, per_head, given):
    """Lists as wide as the cache, of which tiles of rows use a few entries or all."""
    q, k, v = _inputs(1, 2, 4, 400, 3000)
    ids = _lists(1, 8 if per_head else 2, 400, 3000, unit, 1.0)
    counts = torch.full(ids.shape[:3], ids.shape[-1], dtype=torch.int32)
    counts[:, :, :130] = 3
    counts[:, :, 130:256] = 0
    counts[:, :, 300:310] = 1
    if given == "pad":
        ids = torch.where(torch.arange(ids.shape[-1]) < counts[..., None], ids, -1)
        counts = None
    got = _run(dev, q, k, v, ids, unit=unit, counts=counts, out_dtype=torch.float32)
    want = oracle.attend_lists(q, k, v, ids.numpy(), unit=unit,
                               counts=None if counts is None else counts.numpy())
    _check(got, want, 2e-6)


def test_small_calls_and_given_splits_stay_with_the_rows(dev):
    q, k, v = _inputs(1, 2, 4, 300, 1000)
    ids = _lists(1, 8, 300, 1000, 1, 0.6)
    tiles = _run(dev, q, k, v, ids, unit=1, out_dtype=torch.float32)
    rows = _run(dev, q, k, v, ids, unit=1, out_dtype=torch.float32, tiled=False, num_splits=1)
    _check(tiles, rows, 2e-6)
    few = _run(dev, q[:, :, :31], k, v, ids[:, :, :31].contiguous(), unit=1, tiled=None,
               out_dtype=torch.float32)
    _check(few, rows[:, :, :31], 2e-6)


def test_out_may_be_q(dev):
    """Written over q (or over what q starts in), each row is read before it is written,
    rows done again too."""
    q, k, v = _inputs(1, 2, 4, 300, 1000)
    ids = _lists(1, 8, 300, 1000, 1, 0.6)
    ids[:, :, 5::7, 0] = ids[:, :, 5::7, 1]
    kw = dict(unit=1, out_dtype=torch.bfloat16)
    want = _run(dev, q, k, v, ids, **kw)
    qd = q.to(dev)
    got = _run(dev, qd, k, v, ids, unit=1, out=qd, tiled=False)
    _check(got, want, 3e-3)
    both = torch.zeros(1, 8, 300, 256, dtype=torch.bfloat16, device=dev)
    both[..., :128] = q.to(dev)  # side by side: nothing shared
    got = _run(dev, both[..., :128], k, v, ids, unit=1, out=both[..., 128:])
    _check(got, want, 3e-3)
    assert torch.equal(both[..., :128].cpu(), q)
    late = torch.zeros(1, 8, 301, 128, dtype=torch.bfloat16, device=dev)
    late[:, :, 1:] = q.to(dev)  # a query further on: rows of q are other rows of out
    _run(dev, late[:, :, 1:], k, v, ids, unit=1, out=late[:, :, :-1], tiled=False)


def test_tiles_replay_in_a_graph(dev):
    """Captured once, replayed over other inputs between eager calls: lists that run as
    tiles, lists that tiles leave (short, or with a unit twice), and back."""
    q, k, v = _inputs(1, 2, 4, 400, 3000)
    full = _lists(1, 2, 400, 3000, 8, 1.0)
    twice = full.clone()
    twice[:, :, ::3, 5] = twice[:, :, ::3, 6]
    many = torch.full(full.shape[:3], full.shape[-1], dtype=torch.int32)
    cases = [(full, many), (full, torch.full_like(many, 2)), (twice, many // 2), (full, many // 3)]
    want = [oracle.attend_lists(q, k, v, i.numpy(), unit=8, counts=c.numpy()) for i, c in cases]
    qd, kd, vd, ids, counts = (x.to(dev).clone() for x in (q, k, v, *cases[0]))
    _run(dev, qd, kd, vd, ids, unit=8, counts=counts, out_dtype=torch.float32)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sparse_attention(qd, kd, vd, ids, unit=8, counts=counts, out_dtype=torch.float32)
    for i in (0, 1, 2, 3, 1, 0):
        ids.copy_(cases[i][0])
        counts.copy_(cases[i][1])
        out.zero_()
        graph.replay()
        eager = sparse_attention(qd, kd, vd, ids, unit=8, counts=counts, out_dtype=torch.float32)
        _check(out.cpu().double().numpy(), want[i], 2e-6)
        assert torch.equal(out, eager)
