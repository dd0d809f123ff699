"""GPU parity of the read totals (``la_list_reads``) behind the variants' stats:
whole numbers, equal to a count over expanded lists."""

from __future__ import annotations

import copy
import pickle

import pytest
import torch

from linattn_amd.core import AttnConfig
from linattn_amd.registry import build
from linattn_amd.variants import _Totals

pytestmark = pytest.mark.gpu


def _count(ids, unit, offset, t_k):
    tq = ids.shape[2]
    lim = torch.clamp(torch.arange(tq) + offset + 1, max=t_k).view(1, 1, tq, 1)
    n = torch.clamp(lim - ids.long() * unit, min=0, max=unit)
    return float(torch.where(ids >= 0, n, 0).sum(-1).double().mean())


@pytest.mark.parametrize("B,L,tq,W,rep,unit", [(1, 1, 1, 1, 1, 1), (2, 3, 5, 63, 1, 16),
                                               (1, 4, 64, 64, 1, 64), (2, 4, 100, 65, 8, 8),
                                               (3, 8, 257, 9, 1, 64), (1, 2, 700, 130, 1, 1)])
def test_totals_match_a_count(dev, B, L, tq, W, rep, unit):
    g = torch.Generator().manual_seed(W)
    rows = -(-tq // rep)
    t_k = 40 * unit + 3
    ids = torch.randint(-1, 45, (B, L, rows, W), generator=g).to(torch.int32)
    counts = torch.randint(0, W + 1, (B, L, rows), generator=g).to(torch.int32)
    full = ids.repeat_interleave(rep, 2)[:, :, :tq]
    for off in (0, 17 * unit + 2):
        tot = _Totals(ids.to(dev), unit, off, tq, t_k, counts.to(dev), rep=rep)
        assert tot.reads() == _count(full, unit, off, t_k)
        assert tot.counts() == float(counts.double().mean())
    # one list for every query, shared by batch and heads (stride 0)
    one = ids[:1, :1, :1]
    tot = _Totals(one.to(dev).expand(B, L, 1, W), unit, 3, tq, t_k)
    assert tot.reads() == _count(one.expand(B, L, tq, W), unit, 3, t_k)


@pytest.mark.parametrize("name", ["hip_quest", "hip_moba", "hip_xattention", "hip_sliding_window"])
def test_stats_read_when_asked(dev, name):
    """stats() after a forward equals the last chunk's, also from another stream."""
    cfg = AttnConfig(n_heads=4, n_kv_heads=2, head_dim=64, block_size=16, topk_blocks=2, window_size=20)
    q, k, v = (torch.randn(1, h, 100, 64, device=dev) for h in (4, 2, 2))
    m = build(name, cfg)
    _, _, per_chunk = m.forward(q, k, v, chunk=40, collect_stats=True)
    m2 = build(name, cfg)
    m2.forward(q, k, v, chunk=40)
    with torch.cuda.stream(torch.cuda.Stream()):
        assert m2.stats() == per_chunk[-1]
    assert all(isinstance(x, float) for x in m2.stats().values())


def test_copied_and_saved_variants_keep_their_stats(dev):
    cfg = AttnConfig(n_heads=4, n_kv_heads=2, head_dim=64, block_size=16, topk_blocks=2)
    q, k, v = (torch.randn(1, h, 100, 64, device=dev) for h in (4, 2, 2))
    m = build("hip_moba", cfg)
    m.forward(q, k, v)
    assert copy.deepcopy(m).stats() == m.stats()
    assert pickle.loads(pickle.dumps(m)).stats() == m.stats()


@pytest.mark.parametrize("name", ["hip_quest", "hip_moba", "hip_xattention"])
def test_stats_follow_graph_replays(dev, name):
    """Each replay's stats are those of its own inputs, also after stats were read
    before; a copy keeps the numbers it was made with.  (Threshold lists: how many
    blocks a query keeps depends on the values.)"""
    cfg = AttnConfig(n_heads=4, n_kv_heads=2, head_dim=64, block_size=16, topk_blocks=2)
    g = torch.Generator().manual_seed(2)
    ins = [[torch.randn(1, h, 160, 64, generator=g) * s for h in (4, 2, 2)] for s in (0.1, 1.0, 6.0)]
    eager, want = build(name, cfg), []
    for x in ins:
        out, _ = eager.forward(*(t.to(dev) for t in x))
        want.append((out, eager.stats()))
    if name == "hip_xattention":
        assert len({w["blocks_per_query"] for _, w in want}) == len(ins)
    m = build(name, cfg)
    q, k, v = (t.to(dev) for t in ins[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        m.forward(q, k, v)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, _ = m.forward(q, k, v)
    copies = []
    for i in (0, 1, 2, 0, 2):
        for t, x in zip((q, k, v), ins[i]):
            t.copy_(x)
        graph.replay()
        assert m.stats() == want[i][1]
        assert torch.equal(out, want[i][0])
        copies.append((i, copy.deepcopy(m)))
    assert all(c.stats() == want[i][1] for i, c in copies)
