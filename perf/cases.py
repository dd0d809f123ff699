"""The calls whose speed this framework is judged by.

Each case is one call (or the few calls of one step) that a program using
``linattn_amd`` makes through its public entry points: Quest decode over a
paged or contiguous cache, a serving step with append, fp8 decode behind the
lightning indexer, MoBA decode, the indexer's prefill top-k, DSA's chunked
prefill, block-sparse prefill, XAttention's selection, and the prefill of
whole ``hip_*`` variants.

``listed()`` names the cases, ``draw(rng)`` makes another of the same ranges,
``prepare`` builds what the program has in hand, ``run`` is one pass, ``work``
the bytes and operations it cannot do without, ``tolerance`` how far another
correct implementation may be off, ``exact`` the result in 64 bits by plain
torch.
"""

import math

import torch

from linattn_amd.core import AttnConfig
from linattn_amd.kernels.block_sparse import fp8_scale_pairs, sparse_attention
from linattn_amd.kernels.fused_indexer import indexer_topk
from linattn_amd.kernels.kv_cache import paged_kv_append
from linattn_amd.kernels.paged_decode import (indexer_decode_step, quantize_fp8_per_token,
                                              quest_decode_fused, quest_decode_step)
from linattn_amd.kernels.prefill import block_select_hip, block_sparse_prefill, sparse_prefill
from linattn_amd.kernels.quest_pages import page_update_hip, quest_select_hip
from linattn_amd.kernels.routing import block_means_hip, gate_select_hip, xattn_select_hip
from linattn_amd.registry import build

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
_F64 = torch.float64


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # one user, a short context, fp32: the smallest decode step (page scores, top-k,
        # attention), where launches and latency are all there is
        dict(name="quest_small", kind="quest_small", B=1, Hq=8, Hkv=8, T=4096, D=64, page=16,
             topk=16, dtype="fp32"),
        # a serving step of a ragged batch: every sequence appends one token (with its page
        # bounds), selects pages at its own position and attends them
        dict(name="serve_ragged", kind="serve", B=24, Hq=32, Hkv=8, T=6016, D=128, page=64,
             topk=32, dtype="bf16"),
        # long-context decode at a full batch: the headline workload
        dict(name="quest_64k", kind="quest_decode", entry="fused", B=64, Hq=32, Hkv=8, T=65536,
             D=128, page=64, topk=32, dtype="bf16"),
        # fp8 cache of 128K tokens, the lightning indexer picks 4096 of them
        dict(name="fp8_128k", kind="fp8_decode", B=16, Hq=32, Hkv=8, T=131072, D=128, page=64,
             HI=4, d=64, topk=4096, dtype="fp8"),
        # MoBA decode with cached block means
        dict(name="moba_decode", kind="moba_decode", B=16, Hq=32, Hkv=8, T=16384, D=128, block=64,
             topk=16, dtype="bf16"),
        # the lightning indexer over a whole 8K prompt, sorted top-2048 per query
        dict(name="indexer_8k", kind="indexer", B=1, T=8192, HI=4, d=64, topk=2048, dtype="bf16"),
        # chunked prefill with DSA: a chunk of queries at the end of a 16K context, the indexer's
        # token sets and the attention over them
        dict(name="dsa_chunk", kind="dsa_chunk", B=1, Hq=32, Hkv=8, Tq=512, T=16384, D=128, HI=4,
             d=64, topk=2048, dtype="bf16"),
        # block-sparse prefill of two 32K prompts: selection, then attention
        dict(name="block_32k", kind="block_prefill", entry="calls", B=2, Hq=32, Hkv=8, T=32768,
             D=128, ragged=False, dtype="bf16"),
        # a ragged batch of shorter prompts through the one-call prefill with its range check
        dict(name="block_ragged", kind="block_prefill", entry="sparse_prefill", B=3, Hq=16, Hkv=4,
             T=5003, D=128, ragged=True, dtype="bf16"),
        # XAttention's selection at its defaults over an 8K prompt
        dict(name="xattn_8k", kind="xattn", B=1, Hq=32, Hkv=8, T=8192, D=128, block=8, stride=8,
             threshold=0.9, dtype="bf16"),
        # a whole variant over a prompt, at the harness's fp32 configuration and default chunk
        dict(name="quest_prefill", kind="variant", variant="quest", B=2, Hq=4, Hkv=4, T=2048, D=64,
             block=64, topk=4, chunk=0, dtype="fp32"),
        # a whole variant at a model's bf16 configuration: per-query block lists over a 4K prompt
        dict(name="moba_prefill", kind="variant", variant="moba", B=1, Hq=32, Hkv=8, T=4096, D=128,
             block=64, topk=8, chunk=1024, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quest_small", "serve", "quest_decode", "fp8_decode", "moba_decode",
                       "indexer", "dsa_chunk", "block_prefill", "block_prefill", "xattn",
                       "variant", "variant", "variant"])
    heads = rng.choice([(32, 8), (16, 8), (16, 4), (8, 8)])
    if kind == "quest_small":
        H = rng.choice([4, 8, 16])
        return dict(kind=kind, B=rng.randint(1, 4), Hq=H, Hkv=H, T=_log(rng, 256, 8192),
                    D=rng.choice([64, 128]), page=rng.choice([16, 32, 64]),
                    topk=rng.choice([4, 8, 16, 32]), dtype=rng.choice(["fp32", "bf16"]))
    if kind == "serve":
        page = rng.choice([16, 32, 64])
        T = -(-_log(rng, 512, 8192) // page) * page
        return dict(kind=kind, B=_log(rng, 1, 32), Hq=heads[0], Hkv=heads[1], T=T, D=128,
                    page=page, topk=rng.choice([8, 16, 32]), dtype="bf16")
    if kind == "quest_decode":
        page = rng.choice([32, 64])
        B = _log(rng, 1, 64)
        T = -(-_log(rng, 1024, 1024 * page) // page) * page
        return dict(kind=kind, entry="fused" if heads[0] // heads[1] in (2, 4) else "step", B=B,
                    Hq=heads[0], Hkv=heads[1], T=T, D=128, page=page,
                    topk=rng.choice([8, 16, 32, 64]), dtype="bf16")
    if kind == "fp8_decode":
        T = -(-_log(rng, 2048, 131072) // 64) * 64
        return dict(kind=kind, B=_log(rng, 1, 16), Hq=heads[0], Hkv=heads[1], T=T, D=128, page=64,
                    HI=4, d=64, topk=min(T, _log(rng, 256, 4096)), dtype="fp8")
    if kind == "moba_decode":
        return dict(kind=kind, B=_log(rng, 1, 16), Hq=heads[0], Hkv=heads[1],
                    T=_log(rng, 1024, 16384), D=128, block=rng.choice([64, 128]),
                    topk=rng.choice([4, 8, 16]), dtype="bf16")
    if kind == "indexer":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        T = _log(rng, 512, 8192 if dtype == "bf16" else 4096)
        return dict(kind=kind, B=1, T=T, HI=4, d=64, topk=min(T, _log(rng, 64, 2048)), dtype=dtype)
    if kind == "dsa_chunk":
        T = _log(rng, 2048, 16384)
        return dict(kind=kind, B=1, Hq=heads[0], Hkv=heads[1], Tq=_log(rng, 64, 512), T=T, D=128,
                    HI=4, d=64, topk=_log(rng, 256, 2048), dtype="bf16")
    if kind == "block_prefill":
        ragged = rng.random() < 0.4
        return dict(kind=kind, entry=rng.choice(["calls", "sparse_prefill"]), B=rng.randint(1, 2),
                    Hq=heads[0], Hkv=heads[1], T=_log(rng, 700, 8192 if ragged else 32768), D=128,
                    ragged=ragged, dtype="bf16" if rng.random() < 0.7 or ragged else "fp8")
    if kind == "xattn":
        H = rng.choice([(32, 8), (16, 8), (8, 8)])
        return dict(kind=kind, B=1, Hq=H[0], Hkv=H[1], T=_log(rng, 512, 8192), D=128, block=8,
                    stride=8, threshold=rng.choice([0.8, 0.9, 0.95]), dtype="bf16")
    variant = rng.choice(["quest", "moba", "sliding_window"])
    if rng.random() < 0.5:
        return dict(kind=kind, variant=variant, B=rng.randint(1, 2), Hq=8, Hkv=rng.choice([2, 4, 8]),
                    T=_log(rng, 300, 2048), D=64, block=64, topk=rng.choice([4, 8]), chunk=0,
                    dtype="fp32")
    return dict(kind=kind, variant=variant, B=1, Hq=heads[0], Hkv=heads[1], T=_log(rng, 400, 4096),
                D=128, block=64, topk=rng.choice([4, 8]), chunk=rng.choice([0, 512, 1024]),
                dtype="bf16")


# ----------------------------------------------------------------- inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _prompt(g, B, Hq, Hkv, T, D):
    """q, k, v of a prompt: neighbouring tokens share a topic (a direction per KV head that
    a stretch of 128 tokens carries, 24 topics in all), on top of as much noise."""
    stretch = 128
    n = -(-T // stretch)
    topics = _randn(g, B, Hkv, 24, D)
    pick = torch.randint(0, 24, (B, Hkv, n, 1), generator=g, device="cuda").expand(B, Hkv, n, D)
    base = topics.gather(2, pick).repeat_interleave(stretch, 2)[:, :, :T]
    q = 0.7 * base.repeat_interleave(Hq // Hkv, 1) + 0.7 * _randn(g, B, Hq, T, D)
    k = 0.7 * base + 0.7 * _randn(g, B, Hkv, T, D)
    return q, k, _randn(g, B, Hkv, T, D)


def _pool(g, n, Hkv, page, D, dtype, fill=None):
    """Two pools of n pages, filled in pieces (bounded fp32 temporaries)."""
    out = torch.empty(n, Hkv, page, D, dtype=dtype, device="cuda")
    step = 4096
    for i in range(0, n, step):
        x = _randn(g, min(step, n - i), Hkv, page, D)
        if fill is None:
            out[i:i + step] = x
        else:
            fill(out, i, x)
    return out


def _table(g, B, P):
    return torch.randperm(B * P, generator=g, device="cuda").view(B, P).to(torch.int32)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    B = c["B"]
    s = {"case": c}
    if kind == "quest_small":
        dt = _DT[c["dtype"]]
        s["q"] = _randn(g, B, c["Hq"], 1, c["D"]).to(dt)
        s["k"] = _randn(g, B, c["Hkv"], c["T"], c["D"]).to(dt)
        s["v"] = _randn(g, B, c["Hkv"], c["T"], c["D"]).to(dt)
        s["mins"], s["maxs"] = page_update_hip(s["k"], c["page"])
    elif kind in ("serve", "quest_decode"):
        P = c["T"] // c["page"]
        s["q"] = _randn(g, B, c["Hq"], 1, c["D"]).bfloat16()
        s["k_pool"] = _pool(g, B * P, c["Hkv"], c["page"], c["D"], torch.bfloat16)
        s["v_pool"] = _pool(g, B * P, c["Hkv"], c["page"], c["D"], torch.bfloat16)
        s["pt"] = _table(g, B, P)
        lens = None
        if kind == "serve":
            lens = torch.randint(c["T"] // 2, c["T"], (B,), generator=g, device="cuda").to(torch.int32)
            s["positions"] = lens
            s["k_new"] = _randn(g, B, c["Hkv"], 1, c["D"]).bfloat16()
            s["v_new"] = _randn(g, B, c["Hkv"], 1, c["D"]).bfloat16()
        s["mins"], s["maxs"] = page_update_hip(s["k_pool"], c["page"], page_table=s["pt"], kv_len=lens)
    elif kind == "fp8_decode":
        P = c["T"] // c["page"]
        s["q"] = _randn(g, B, c["Hq"], 1, c["D"]).bfloat16()
        ks, vs = fp8_scale_pairs(B * P, c["Hkv"], c["page"], "cuda")

        def into(scales):
            def put(out, i, x):
                out[i:i + x.shape[0]], scales[i:i + x.shape[0]] = quantize_fp8_per_token(x)
            return put

        s["k_pool"] = _pool(g, B * P, c["Hkv"], c["page"], c["D"], torch.float8_e4m3fn, into(ks))
        s["v_pool"] = _pool(g, B * P, c["Hkv"], c["page"], c["D"], torch.float8_e4m3fn, into(vs))
        s["k_scale"], s["v_scale"] = ks, vs
        s["pt"] = _table(g, B, P)
        s["q_idx"] = _randn(g, B, 1, c["HI"], c["d"]).bfloat16()
        s["k_idx"] = _randn(g, B, c["T"], c["HI"], c["d"]).bfloat16()
        s["w"] = torch.rand(B, 1, c["HI"], generator=g, device="cuda")
    elif kind == "moba_decode":
        q, k, v = _prompt(g, B, c["Hq"], c["Hkv"], c["T"], c["D"])
        s["q"], s["k"], s["v"] = q[:, :, -1:].bfloat16(), k.bfloat16(), v.bfloat16()
        s["kbar"] = block_means_hip(s["k"], block=c["block"])
        s["newest"] = torch.full((B,), c["T"] - 1, dtype=torch.int32, device="cuda")
    elif kind in ("indexer", "dsa_chunk"):
        dt, Tq = _DT[c["dtype"]], c.get("Tq", c["T"])
        s["q_idx"] = _randn(g, B, Tq, c["HI"], c["d"]).to(dt)
        s["k_idx"] = _randn(g, B, c["T"], c["HI"], c["d"]).to(dt)
        s["w"] = torch.rand(B, Tq, c["HI"], generator=g, device="cuda")
        if kind == "dsa_chunk":
            s["q"] = _randn(g, B, c["Hq"], Tq, c["D"]).to(dt)
            s["k"] = _randn(g, B, c["Hkv"], c["T"], c["D"]).to(dt)
            s["v"] = _randn(g, B, c["Hkv"], c["T"], c["D"]).to(dt)
    elif kind == "block_prefill":
        T = c["T"]
        q = _randn(g, B, c["Hq"], T, c["D"])
        k = _randn(g, B, c["Hkv"], T, c["D"])
        v = _randn(g, B, c["Hkv"], T, c["D"])
        # one key in a hundred is an outlier, as attention sinks and rare tokens are
        k *= 1.0 + 7.0 * (torch.rand(B, c["Hkv"], T, 1, generator=g, device="cuda") < 0.01)
        s["q"] = q.bfloat16()
        s["k"], s["v"] = k.bfloat16(), v.bfloat16()
        if c["dtype"] == "fp8":  # the selection reads bf16 keys, the attention the fp8 cache
            s["kc"], s["ks"] = quantize_fp8_per_token(k)
            s["vc"], s["vs"] = quantize_fp8_per_token(v)
        if c["ragged"]:
            lens = torch.randint(T // 8, T, (B,), generator=g, device="cuda").to(torch.int32)
            lens[0] = T
            s["lengths"] = lens
    elif kind == "xattn":
        q, k, _ = _prompt(g, B, c["Hq"], c["Hkv"], c["T"], c["D"])
        s["q"], s["k"] = q.bfloat16(), k.bfloat16()
    else:  # variant
        dt = _DT[c["dtype"]]
        s["q"], s["k"], s["v"] = (x.to(dt) for x in _prompt(g, B, c["Hq"], c["Hkv"], c["T"], c["D"]))
        cfg = AttnConfig(n_heads=c["Hq"], n_kv_heads=c["Hkv"], head_dim=c["D"],
                         block_size=c["block"], topk_blocks=c["topk"], dtype=dt)
        s["model"] = build("hip_" + c["variant"], cfg)
    return s


# ---------------------------------------------------------------- one pass ----
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "quest_small":
        ids, counts = quest_select_hip(s["q"], s["mins"], s["maxs"], page_size=c["page"],
                                       topk=c["topk"], offset=c["T"] - 1)
        out = sparse_attention(s["q"], s["k"], s["v"], ids, unit=c["page"], counts=counts,
                               causal=True, offset=c["T"] - 1)
        return {"out": out, "ids": ids, "counts": counts}
    if kind == "serve":
        paged_kv_append(s["k_new"], s["v_new"], s["k_pool"], s["v_pool"], s["pt"], s["positions"],
                        page_min=s["mins"], page_max=s["maxs"], page_size=c["page"])
        out, ids, counts = quest_decode_step(s["q"], s["k_pool"], s["v_pool"], s["pt"], s["mins"],
                                             s["maxs"], page_size=c["page"], topk=c["topk"],
                                             positions=s["positions"])
        return {"out": out, "ids": ids, "counts": counts, "k_pool": s["k_pool"],
                "v_pool": s["v_pool"], "mins": s["mins"], "maxs": s["maxs"]}
    if kind == "quest_decode":
        step = quest_decode_fused if c["entry"] == "fused" else quest_decode_step
        out, ids, counts = step(s["q"], s["k_pool"], s["v_pool"], s["pt"], s["mins"], s["maxs"],
                                page_size=c["page"], topk=c["topk"], pos=c["T"] - 1)
        return {"out": out, "ids": ids, "counts": counts}
    if kind == "fp8_decode":
        out, ids = indexer_decode_step(s["q"], s["k_pool"], s["v_pool"], s["pt"], s["q_idx"],
                                       s["k_idx"], s["w"], topk=c["topk"], pos=c["T"] - 1,
                                       page_size=c["page"], k_scale=s["k_scale"],
                                       v_scale=s["v_scale"])
        return {"out": out, "ids": ids}
    if kind == "moba_decode":
        block_means_hip(s["k"], block=c["block"], out=s["kbar"], positions=s["newest"])
        ids, counts = gate_select_hip(s["q"], s["k"], block=c["block"], topk=c["topk"],
                                      offset=c["T"] - 1, kbar=s["kbar"])
        out = sparse_attention(s["q"], s["k"], s["v"], ids, unit=c["block"], counts=counts,
                               causal=True, offset=c["T"] - 1)
        return {"out": out, "ids": ids, "counts": counts, "kbar": s["kbar"]}
    if kind == "indexer":
        val, idx = indexer_topk(s["q_idx"], s["k_idx"], s["w"], c["topk"], causal=True)
        return {"val": val, "idx": idx}
    if kind == "dsa_chunk":
        off = c["T"] - c["Tq"]
        _, idx = indexer_topk(s["q_idx"], s["k_idx"], s["w"], c["topk"], causal=True, offset=off,
                              sorted=False)
        ids = idx.unsqueeze(1).expand(c["B"], c["Hkv"], c["Tq"], idx.shape[-1])
        out = sparse_attention(s["q"], s["k"], s["v"], ids, unit=1, causal=True, offset=off)
        return {"out": out, "idx": idx}
    if kind == "block_prefill":
        if c["entry"] == "sparse_prefill" and c["dtype"] == "bf16":
            out, ids, counts = sparse_prefill(s["q"], s["k"], s["v"], lengths=s.get("lengths"))
            return {"out": out, "ids": ids, "counts": counts}
        ids, counts = block_select_hip(s["q"], s["k"], lengths=s.get("lengths"))
        if c["dtype"] == "fp8":
            out = block_sparse_prefill(s["q"], s["kc"], s["vc"], ids, counts, k_scale=s["ks"],
                                       v_scale=s["vs"], check_range=False)
        else:
            out = block_sparse_prefill(s["q"], s["k"], s["v"], ids, counts, check_range=False,
                                       lengths=s.get("lengths"))
        return {"out": out, "ids": ids, "counts": counts}
    if kind == "xattn":
        ids, counts = xattn_select_hip(s["q"], s["k"], block=c["block"], stride=c["stride"],
                                       threshold=c["threshold"])
        return {"ids": ids, "counts": counts}
    out, state = s["model"].forward(s["q"], s["k"], s["v"], chunk=c["chunk"] or None)
    return {"out": out, **{n: t for n, t in sorted(state.items()) if isinstance(t, torch.Tensor)}}


# ------------------------------------------------------------------- work ----
def _union(n, k, heads):
    """Expected size of the union of `heads` lists of k out of n, drawn independently."""
    return n * (1.0 - (1.0 - min(k, n) / n) ** heads)


def _kept(T, first, budget):
    """Sum over positions first .. T-1 of the tokens a query reads: its prefix, at most budget."""
    return sum(min(budget, t + 1) for t in range(first, T))


def work(case):
    c, kind, B = case, case["kind"], case["B"]
    esz = {"bf16": 2, "fp32": 4, "fp8": 1}[c["dtype"]]
    if kind in ("quest_small", "serve", "quest_decode"):
        P = -(-c["T"] // c["page"])
        vis = P if kind != "serve" else 0.75 * P
        G = c["Hq"] // c["Hkv"]
        pages = min(vis, _union(vis, min(c["topk"], vis), G))
        kv = B * c["Hkv"] * pages * c["page"] * c["D"] * 2 * esz
        meta = B * c["Hkv"] * vis * c["D"] * 2 * esz
        flops = B * c["Hq"] * c["D"] * (4 * pages * c["page"] + 4 * vis)
        new = B * c["Hkv"] * c["D"] * esz * 8 if kind == "serve" else 0
        return {"bytes": kv + meta + new + 2 * B * c["Hq"] * c["D"] * esz
                + 4 * B * c["Hkv"] * G * c["topk"], "flops": flops}
    if kind == "fp8_decode":
        return {"bytes": B * c["T"] * c["HI"] * c["d"] * 2
                + B * c["Hkv"] * c["topk"] * (2 * c["D"] + 8) + 4 * B * c["Hq"] * c["D"],
                "flops": 2 * B * c["T"] * c["HI"] * c["d"] + 4 * B * c["Hq"] * c["topk"] * c["D"]}
    if kind == "moba_decode":
        nkb = -(-c["T"] // c["block"])
        blocks = _union(nkb, c["topk"] + 1, c["Hq"] // c["Hkv"])
        return {"bytes": B * c["Hkv"] * (8 * nkb * c["D"] + blocks * c["block"] * c["D"] * 4)
                + 4 * B * c["Hq"] * c["D"],
                "flops": B * c["Hq"] * c["D"] * (2 * nkb + 4 * (c["topk"] + 1) * c["block"])}
    if kind == "indexer":
        pairs = c["T"] * (c["T"] + 1) // 2
        return {"bytes": B * c["T"] * (2 * c["HI"] * c["d"] * esz + 4 * c["HI"] + 8 * c["topk"]),
                "flops": B * pairs * c["HI"] * (2 * c["d"] + 3)}
    if kind == "dsa_chunk":
        Tq, T = c["Tq"], c["T"]
        pairs = Tq * (T - Tq) + Tq * (Tq + 1) // 2
        kept = _kept(T, T - Tq, c["topk"])
        return {"bytes": B * ((Tq + T) * c["HI"] * c["d"] * 2 + 4 * Tq * c["topk"]
                              + 2 * c["Hkv"] * T * c["D"] * 2 + 2 * c["Hq"] * Tq * c["D"] * 2),
                "flops": B * (pairs * c["HI"] * 2 * c["d"] + 4 * c["Hq"] * c["D"] * kept)}
    if kind == "block_prefill":
        T, bs = c["T"], 64
        nqb = -(-T // bs)
        pairs = sum(min(qb + 1, 21) for qb in range(nqb)) * bs * bs
        share = 1.0 if not c["ragged"] else (1.0 + (B - 1) * 0.56) / B
        kv = 2 * B * c["Hkv"] * T * c["D"] * (2 if c["dtype"] == "bf16" else 3)
        return {"bytes": share * (kv + 4 * B * c["Hq"] * T * c["D"] + 4 * B * c["Hq"] * nqb * 21),
                "flops": share * B * c["Hq"] * (4 * c["D"] * pairs + c["D"] * nqb * nqb)}
    if kind == "xattn":
        n = -(-c["T"] // c["block"])
        return {"bytes": B * (c["Hq"] + c["Hkv"]) * c["T"] * c["D"] * 2 + 4 * B * c["Hq"] * n * n,
                "flops": B * c["Hq"] * n * (n + 1) // 2 * c["block"] * c["D"] * 2}
    T, D = c["T"], c["D"]
    if c["variant"] == "sliding_window":
        kept, sel = _kept(T, 0, 256 + 4), 0
    else:
        nb = -(-T // c["block"])
        budget = (c["topk"] + (c["variant"] == "moba")) * c["block"]
        kept, sel = _kept(T, 0, budget), (4 if c["variant"] == "quest" else 2) * D * T * nb // 2
    return {"bytes": B * T * D * esz * (2 * c["Hq"] + 4 * c["Hkv"]),
            "flops": B * c["Hq"] * (4 * D * kept + sel)}


# -------------------------------------------------------------- tolerance ----
def tolerance(case):
    """Selections and stored bytes are whole values and stay the same; scores are exact sums
    rounded once.  Outputs: fp32 ones are fp32 sums, bf16 ones a rounding to 8 bits."""
    if case["kind"] in ("indexer", "xattn"):
        return "exact"
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    return {"rel": 7e-3}


# ------------------------------------------------------------------ exact ----
def _softmax_rows(x):
    """Softmax over the last dim of fp64 scores; a row without a finite score is zeros."""
    m = x.amax(-1, keepdim=True)
    m = torch.where(torch.isfinite(m), m, torch.zeros_like(m))
    e = torch.exp(x - m)
    s = e.sum(-1, keepdim=True)
    return e / torch.where(s > 0, s, torch.ones_like(s))


def _quest_pages(q, mins, maxs, pos, page, topk):
    """Boolean (H, P): the pages each query head of one sequence keeps.  q (H, D), bounds
    (H, P, D) in fp64."""
    P = mins.shape[1]
    sc = torch.maximum(q[:, None] * mins, q[:, None] * maxs).sum(-1)
    start = torch.arange(P, device=q.device) * page
    sc = sc.masked_fill(start > pos, float("-inf"))
    sc[:, min(pos // page, P - 1)] = float("inf")
    order = torch.sort(sc, dim=-1, descending=True, stable=True).indices[:, :max(1, min(topk, P))]
    keep = torch.zeros_like(sc, dtype=torch.bool).scatter_(1, order, True)
    return keep & (start <= pos)


def _bounds(k, page):
    """(Hkv, P, D) minima and maxima of k (Hkv, T, D) per page."""
    H, T, D = k.shape
    P = -(-T // page)
    lo = torch.full((H, P * page, D), float("inf"), dtype=_F64, device=k.device)
    hi = torch.full_like(lo, float("-inf"))
    lo[:, :T], hi[:, :T] = k, k
    return lo.view(H, P, page, D).amin(2), hi.view(H, P, page, D).amax(2)


def _decode_masked(q, k, v, mask):
    """q (H, D), k and v (Hkv, T, D), mask (H, T): the attention of one query, fp64."""
    H, D = q.shape
    G = H // k.shape[0]
    x = torch.matmul(q.view(-1, G, D), k.transpose(1, 2)) / math.sqrt(D)
    x = x.masked_fill(~mask.view(-1, G, mask.shape[-1]), float("-inf"))
    return torch.matmul(_softmax_rows(x), v).reshape(H, D)


def _exact_quest(case, s):
    c = case
    H, G = c["Hq"], c["Hq"] // c["Hkv"]
    out = torch.empty(c["B"], H, 1, c["D"], dtype=_F64, device="cuda")
    for b in range(c["B"]):
        if "pt" in s:
            rows = s["pt"][b].long()
            k = s["k_pool"][rows].transpose(0, 1).reshape(c["Hkv"], -1, c["D"]).to(_F64)
            v = s["v_pool"][rows].transpose(0, 1).reshape(c["Hkv"], -1, c["D"]).to(_F64)
        else:
            k, v = s["k"][b].to(_F64), s["v"][b].to(_F64)
        pos = c["T"] - 1
        if "positions" in s:
            pos = int(s["positions"][b])
            k[:, pos], v[:, pos] = s["k_new"][b, :, 0].to(_F64), s["v_new"][b, :, 0].to(_F64)
            k, v = k[:, :pos + 1], v[:, :pos + 1]
        q = s["q"][b, :, 0].to(_F64)
        lo, hi = _bounds(k, c["page"])
        keep = torch.cat([_quest_pages(q[h:h + 1], lo[h // G:h // G + 1], hi[h // G:h // G + 1],
                                       pos, c["page"], c["topk"]) for h in range(H)])
        if G > 1:
            keep = keep.view(-1, G, keep.shape[1]).any(1, keepdim=True)
            keep = keep.expand(-1, G, -1).reshape(H, -1)
        mask = keep.repeat_interleave(c["page"], 1)[:, :k.shape[1]]
        out[b, :, 0] = _decode_masked(q, k, v, mask)
    return out


def _indexer_scores(s, t0, t1, offset):
    """fp64 scores (B, t1-t0, T) of queries t0 .. t1-1, -inf past each query's position."""
    q, k, w = s["q_idx"][:, t0:t1].to(_F64), s["k_idx"].to(_F64), s["w"][:, t0:t1].to(_F64)
    T = k.shape[1]
    x = torch.zeros(q.shape[0], t1 - t0, T, dtype=_F64, device="cuda")
    for h in range(q.shape[2]):
        x += w[:, :, h, None] * torch.relu(torch.matmul(q[:, :, h], k[:, :, h].transpose(1, 2)))
    pos = torch.arange(t0, t1, device="cuda") + offset
    return x.masked_fill(torch.arange(T, device="cuda") > pos[:, None], float("-inf"))


def _top_mask(x, k):
    order = torch.sort(x, dim=-1, descending=True, stable=True).indices[..., :k]
    keep = torch.zeros_like(x, dtype=torch.bool).scatter_(-1, order, True)
    return keep & torch.isfinite(x)


def _exact_fp8(c, s):
    out = torch.empty(c["B"], c["Hq"], 1, c["D"], dtype=_F64, device="cuda")
    keep = _top_mask(_indexer_scores(s, 0, 1, c["T"] - 1)[:, 0], c["topk"])
    for b in range(c["B"]):
        tok = torch.nonzero(keep[b])[:, 0]
        rows, at = s["pt"][b].long()[tok // c["page"]], tok % c["page"]
        k = s["k_pool"][rows, :, at].to(_F64) * s["k_scale"][rows, :, at].to(_F64)[..., None]
        v = s["v_pool"][rows, :, at].to(_F64) * s["v_scale"][rows, :, at].to(_F64)[..., None]
        mask = torch.ones(c["Hq"], len(tok), dtype=torch.bool, device="cuda")
        out[b, :, 0] = _decode_masked(s["q"][b, :, 0].to(_F64), k.transpose(0, 1),
                                      v.transpose(0, 1), mask)
    return out


def _means(k, block):
    """(H, blocks, D) fp64 block means, the last block padded by repeating its last row."""
    H, T, D = k.shape
    n = -(-T // block)
    k = torch.cat([k, k[:, -1:].expand(H, n * block - T, D)], 1)
    return k.view(H, n, block, D).mean(2)


def _moba_blocks(q, kbar, pos, block, topk):
    """Boolean (Hq, Tq, blocks) of q (Hq, Tq, D) at positions pos (Tq,)."""
    H, n = q.shape[0], kbar.shape[1]
    gate = torch.matmul(q, kbar.repeat_interleave(H // kbar.shape[0], 0).transpose(1, 2))
    start = torch.arange(n, device=q.device) * block
    keep = _top_mask(gate.masked_fill(start > pos[:, None], float("-inf")), topk)
    own = torch.arange(n, device=q.device) == (pos // block)[:, None]
    return keep | own


def _exact_block_prefill(c, s):
    B, G, T, D, bs = c["B"], c["Hq"] // c["Hkv"], c["T"], c["D"], 64
    out = torch.zeros(B, c["Hq"], T, D, dtype=_F64, device="cuda")
    for b in range(B):
        L = int(s["lengths"][b]) if "lengths" in s else T
        n = -(-L // bs)
        qb = torch.arange(n, device="cuda")
        causal = qb[None, :] <= qb[:, None]
        fixed = ((qb[None, :] < 1) | (qb[None, :] > qb[:, None] - 4)) & causal
        for h in range(c["Hq"]):
            q, k, v = s["q"][b, h, :L].to(_F64), s["k"][b, h // G, :L].to(_F64), None
            sc = torch.matmul(_means(q[None], bs)[0], _means(k[None], bs)[0].T)
            keep = _top_mask(sc.masked_fill(~causal, float("-inf")), 16) | fixed
            if c["dtype"] == "fp8":
                k = s["kc"][b, h // G].to(_F64) * s["ks"][b, h // G].to(_F64)[:, None]
                v = s["vc"][b, h // G].to(_F64) * s["vs"][b, h // G].to(_F64)[:, None]
            else:
                v = s["v"][b, h // G, :L].to(_F64)
            pad = n * bs - L
            k, v, q = (torch.nn.functional.pad(x, (0, 0, 0, pad)).view(n, bs, D) for x in (k, v, q))
            W = int(keep.sum(1).max())
            lst = torch.sort(keep.to(torch.int8), dim=1, descending=True, stable=True).indices[:, :W]
            there = torch.gather(keep, 1, lst)
            for i in range(0, n, 128):
                j = slice(i, min(i + 128, n))
                kk, vv = k[lst[j]].flatten(1, 2), v[lst[j]].flatten(1, 2)
                tok = (lst[j][:, :, None] * bs + torch.arange(bs, device="cuda")).flatten(1)
                row = qb[j][:, None] * bs + torch.arange(bs, device="cuda")
                ok = (tok[:, None] <= row[:, :, None]) & there[j].repeat_interleave(bs, 1)[:, None]
                x = torch.matmul(q[j], kk.transpose(1, 2)) / math.sqrt(D)
                o = torch.matmul(_softmax_rows(x.masked_fill(~ok, float("-inf"))), vv).flatten(0, 1)
                end = min(L, i * bs + o.shape[0])
                out[b, h, i * bs:end] = o[:end - i * bs]
    return out


def _exact_variant(c, s):
    """The whole prompt at once: every chunk is a multiple of the block, so a query's blocks
    are complete up to its chunk's end and the chunks change nothing."""
    B, G, T, D, bs = c["B"], c["Hq"] // c["Hkv"], c["T"], c["D"], c["block"]
    out = torch.empty(B, c["Hq"], T, D, dtype=_F64, device="cuda")
    pos = torch.arange(T, device="cuda")
    causal = pos[None, :] <= pos[:, None]
    for b in range(B):
        for kvh in range(c["Hkv"]):
            k, v = s["k"][b, kvh].to(_F64), s["v"][b, kvh].to(_F64)
            q = s["q"][b, kvh * G:(kvh + 1) * G].to(_F64)
            if c["variant"] == "moba":
                keep = _moba_blocks(q, _means(k[None], bs), pos, bs, c["topk"])
            elif c["variant"] == "quest":
                lo, hi = _bounds(k[None], bs)
                n = lo.shape[1]
                start = torch.arange(n, device="cuda") * bs
                sc = (torch.matmul(torch.relu(q), hi[0].T) - torch.matmul(torch.relu(-q), lo[0].T))
                sc = sc.masked_fill(start > pos[:, None], float("-inf"))
                own = torch.arange(n, device="cuda") == (pos // bs)[:, None]
                keep = _top_mask(sc.masked_fill(own, 1e300), max(1, min(c["topk"], n)))
                keep = keep.any(0, keepdim=True).expand(G, -1, -1)
            else:
                keep = None
            for g in range(G):
                if keep is None:
                    ok = causal & ((pos[None, :] > pos[:, None] - 256) | (pos[None, :] < 4))
                else:
                    ok = causal & keep[g].repeat_interleave(bs, 1)[:, :T]
                x = (torch.matmul(q[g], k.T) / math.sqrt(D)).masked_fill(~ok, float("-inf"))
                out[b, kvh * G + g] = torch.matmul(_softmax_rows(x), v)
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "xattn":
        return None  # whole values only
    s = prepare(case, seed)
    if kind in ("quest_small", "quest_decode"):
        return {"out": _exact_quest(c, s), "ids": None, "counts": None}
    if kind == "serve":
        return {"out": _exact_quest(c, s), "ids": None, "counts": None, "k_pool": None,
                "v_pool": None, "mins": None, "maxs": None}
    if kind == "fp8_decode":
        return {"out": _exact_fp8(c, s), "ids": None}
    if kind == "moba_decode":
        out, pos = [], torch.tensor([c["T"] - 1], device="cuda")
        for b in range(c["B"]):
            k, v, q = s["k"][b].to(_F64), s["v"][b].to(_F64), s["q"][b].to(_F64)
            keep = _moba_blocks(q, _means(k, c["block"]), pos, c["block"], c["topk"])[:, 0]
            mask = keep.repeat_interleave(c["block"], 1)[:, :c["T"]]
            out.append(_decode_masked(q[:, 0], k, v, mask)[None, :, None])
        return {"out": torch.cat(out), "ids": None, "counts": None, "kbar": None}
    if kind == "indexer":
        val = [torch.topk(_indexer_scores(s, t, min(t + 2048, c["T"]), 0), c["topk"], dim=-1).values
               for t in range(0, c["T"], 2048)]
        return {"val": torch.cat(val, 1), "idx": None}
    if kind == "dsa_chunk":
        off, out = c["T"] - c["Tq"], []
        for b in range(c["B"]):
            sb = {n: s[n][b:b + 1] for n in ("q_idx", "k_idx", "w")}
            keep = _top_mask(_indexer_scores(sb, 0, c["Tq"], off)[0], min(c["topk"], c["T"]))
            k, v, q = s["k"][b].to(_F64), s["v"][b].to(_F64), s["q"][b].to(_F64)
            G = c["Hq"] // c["Hkv"]
            for h in range(c["Hq"]):
                x = torch.matmul(q[h], k[h // G].T) / math.sqrt(c["D"])
                out.append(torch.matmul(_softmax_rows(x.masked_fill(~keep, float("-inf"))), v[h // G]))
        return {"out": torch.stack(out).view(c["B"], c["Hq"], c["Tq"], c["D"]), "idx": None}
    if kind == "block_prefill":
        return {"out": _exact_block_prefill(c, s), "ids": None, "counts": None}
    keys = {"quest": ("k", "page_max", "page_min", "v"), "moba": ("block_means", "k", "v"),
            "sliding_window": ("k", "v")}[c["variant"]]
    return {"out": _exact_variant(c, s), **{n: None for n in keys}}
