"""XAttention's slots on the int8 matrix cores against the fp64 form.

Both are exact sums in the same order, so the block lists must be identical, bit
for bit.  A workspace of one run of 64 query blocks' slots has no room for limbs and
takes the fp64 form.  The data decide what a pair takes: an exponent range within
the bound (int8), a few rows past it (listed pairs), most rows past it (tiles left
to the fp64 kernel), infs and NaN."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # B, Hq, Hkv, Tq, T, D, block, offset: from 256 key blocks and 512 tiles on
    (1, 32, 8, 2048, 2048, 128, 8, 0),     # whole tiles; heads spread over XCDs
    (2, 18, 2, 1030, 1030, 128, 4, 0),     # a partial last block and tile
    (1, 36, 4, 530, 530, 64, 2, 0),
    (2, 32, 8, 650, 2600, 64, 8, 1950),    # queries at an offset
    (2, 28, 4, 1030, 4110, 128, 16, 3080),  # the largest block
]


def _inputs(shape, data):
    B, Hq, Hkv, Tq, T, D, blk, off = shape
    g = torch.Generator().manual_seed(T + D)
    q = torch.randn(B, Tq, Hq, D, generator=g)
    k = torch.randn(B, Hkv, T, D, generator=g)
    if data == "few":  # rows of more than 23 octaves
        q[:, 5::97, :, 0] = 3e7
        k[:, :, 11::131, -1] = 1e-9
    elif data == "wide":
        q *= torch.exp(4 * torch.randn(q.shape, generator=g))
        k *= torch.exp(4 * torch.randn(k.shape, generator=g))
    elif data == "special":
        q[:, 17] = 0.0
        q[:, 30, :, 3] = float("inf")
        k[:, :, 40, 5] = float("nan")
        k[:, :, 41, 6] = -float("inf")
        k[:, :, 50] = 1e-40  # denormal
    # [B, Hq, Tq, D] over [B, Tq, Hq, D]
    return q.bfloat16().cuda().transpose(1, 2), k.bfloat16().cuda()


def _select(q, k, **kw):
    """ids, counts and the workspace bytes the library asked for."""
    from linattn_amd import _native as N
    from linattn_amd.kernels.routing import xattn_select_hip
    lib, seen = N.load(), []
    orig = lib.la_xattn_select_workspace

    def workspace(a):
        seen.append(orig(a))
        return seen[-1]

    lib.la_xattn_select_workspace = workspace
    try:
        ids, counts = xattn_select_hip(q, k, **kw)
    finally:
        lib.la_xattn_select_workspace = orig
    return ids, counts, seen[0]


def _slot_bytes(shape, n_qb):
    return shape[0] * shape[1] * n_qb * -(-shape[4] // shape[6]) * 2 * 8


@pytest.mark.parametrize("data", ["normal", "few", "wide", "special"])
@pytest.mark.parametrize("shape", SHAPES)
def test_int8_slots_select_as_fp64(shape, data):
    B, Hq, Hkv, Tq, T, D, blk, off = shape
    q, k = _inputs(shape, data)
    for sel in (dict(threshold=0.9), dict(topk=7)):
        kw = dict(block=blk, stride=blk, offset=off, **sel)
        ids, counts, ws = _select(q, k, **kw)
        # slots of every query block, and the limbs of k and q beside them: the int8 form
        assert ws > _slot_bytes(shape, -(-Tq // blk)) + 4 * D * B * (Hkv * T + Hq * Tq)
        rids, rcounts, _ = _select(q, k, max_workspace_bytes=_slot_bytes(shape, 64), **kw)
        assert torch.equal(counts, rcounts)
        assert torch.equal(ids, rids)


@pytest.mark.parametrize("data", ["normal", "few", "special"])
@pytest.mark.parametrize("chunk", [64, 128])
def test_int8_slots_in_chunks(chunk, data):
    """Two or three chunks of query blocks, the last one partial (its limbs in buffers
    laid out for a whole one): the workspace of a call of one chunk's queries is what
    such a chunk takes, limbs included."""
    shape = (2, 28, 4, 201 * 4 - 1, 1030, 64, 4, 230)
    B, Hq, Hkv, Tq, T, D, blk, off = shape
    q, k = _inputs(shape, data)
    for sel in (dict(threshold=0.9), dict(topk=7)):
        kw = dict(block=blk, stride=blk, offset=off, **sel)
        one = q[:, :, :128 * blk]  # (512 tiles need two rows of them)
        ws = _select(one, k, **kw)[2]
        limbs = ws - _slot_bytes(shape, 128)
        assert limbs > 4 * D * B * (Hkv * T + Hq * 128 * blk)
        if chunk == 64:  # half the slots, half the limbs of q
            ws -= _slot_bytes(shape, 64) + 4 * D * B * Hq * 64 * blk
        ids, counts, full = _select(q, k, max_workspace_bytes=ws, **kw)
        assert full > ws  # more than one chunk
        rids, rcounts, _ = _select(q, k, max_workspace_bytes=_slot_bytes(shape, 64), **kw)
        assert torch.equal(counts, rcounts)
        assert torch.equal(ids, rids)
        whole, wcounts, _ = _select(q, k, **kw)
        assert torch.equal(counts, wcounts) and torch.equal(ids, whole)


@pytest.mark.parametrize("data", ["equal", "levels", "normal", "steep"])
@pytest.mark.parametrize("n_kb", [1, 64, 65, 130, 300, 1000])
def test_threshold_search_of_one_wave(n_kb, data):
    """The wave's search (bits, then the last 64 blocks at once) keeps what the
    workgroup's bitwise search keeps: more than 64 equal masses (never down to a
    block per lane), a few levels of equal masses, and no two equal."""
    from linattn_amd.kernels.routing import xattn_select_hip
    g = torch.Generator().manual_seed(n_kb)
    q = torch.randn(1, 2, 2 * n_kb, 16, generator=g)
    k = torch.randn(1, 1, 2 * n_kb, 16, generator=g)
    if data == "equal":
        q.zero_()
    elif data == "levels":
        q.fill_(0.5)
        k = torch.randint(0, 3, (1, 1, 2 * n_kb, 1), generator=g).float().expand(k.shape).contiguous()
    elif data == "steep":
        q *= 20
    q, k = q.half().cuda(), k.half().cuda()
    for thr in (0.02, 0.5, 0.9, 0.9999999, 1.0):
        kw = dict(block=2, stride=2, threshold=thr)
        ids, counts = xattn_select_hip(q, k, **kw)
        rids, rcounts = xattn_select_hip(q, k, max_workspace_bytes=0, **kw)
        assert torch.equal(counts, rcounts)
        assert torch.equal(ids, rids)
