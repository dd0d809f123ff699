"""Host-side logic that needs no GPU: the variant registry and contract, the
no-fallback rule, and argument validation of the kernel wrappers."""

from __future__ import annotations

import pytest
import torch

from linattn_amd.core import AttnConfig
from linattn_amd.kernels import backend_for, describe_backends
from linattn_amd.kernels.block_sparse import block_sparse_attention, sparse_attention
from linattn_amd.kernels.fused_indexer import indexer_topk
from linattn_amd.kernels.quest_pages import alloc_page_meta, page_select_hip
from linattn_amd.registry import KERNEL_VARIANTS, build, describe_kernel


def test_registry_names_and_errors():
    """registry.py:225-236: <backend>_<variant> names, KeyError otherwise."""
    assert set(KERNEL_VARIANTS) == {"hip_quest", "hip_dsa", "hip_moba", "hip_xattention",
                                    "hip_sliding_window", "hip_streaming_sink"}
    assert describe_kernel("hip_xattention")["reference"] == "xattention"
    # the three selection rules of selection.py:578-590; anything else is refused
    for mode in ("threshold", "topk", "top_ratio"):
        assert build("hip_xattention", extras={"select_mode": mode}).select_mode == mode
    with pytest.raises(ValueError):
        build("hip_xattention", extras={"select_mode": "top_p"})
    assert describe_kernel("hip_moba")["reference"] == "moba"
    assert describe_kernel("hip_quest")["reference"] == "quest"
    assert build("hip_quest").name == "hip_quest"
    with pytest.raises(KeyError):
        build("hip_nope")
    with pytest.raises(KeyError):
        describe_kernel("quest")


def test_config_contract():
    """core.py:47-78 field names, group size, unknown-field and GQA errors."""
    c = AttnConfig(n_heads=8, n_kv_heads=2)
    assert c.group_size == 4 and c.with_(topk_blocks=9).topk_blocks == 9
    with pytest.raises(TypeError):
        build("hip_quest", AttnConfig(), not_a_field=1)
    with pytest.raises(ValueError):
        build("hip_quest", AttnConfig(n_heads=3, n_kv_heads=2))


def test_cost_model_follows_the_reference_conventions():
    """read_budget / flops / memory_bytes of the torch variants
    (selection.py:118-133, local.py:55-61)."""
    c = AttnConfig(n_heads=4, n_kv_heads=2, head_dim=64, block_size=16, window_size=32,
                   topk_blocks=3, sink_size=2)
    q = build("hip_quest", c)
    assert q.read_budget(1000) == 3 * 16 + 32
    n_pages = (1000 + 15) // 16
    assert q.flops(1000) == 4 * 4 * 1000 * 80 * 64 + 2 * 4 * 1000 * n_pages * 64
    w = build("hip_sliding_window", c)
    assert w.read_budget(1000) == 34 and w.memory_bytes(1000) == 2 * 34 * 64 * 4


def test_cpu_tensors_are_rejected_not_served_on_cpu():
    """There is no CPU fallback (the oracle is not a backend)."""
    q = torch.randn(1, 2, 1, 64)
    k = torch.randn(1, 2, 32, 64)
    ids = torch.zeros(1, 2, 1, 1, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="GPU"):
        sparse_attention(q, k, k, ids, unit=16)
    with pytest.raises(RuntimeError, match="GPU"):
        block_sparse_attention(q, k, k, ids, block_size=16)
    with pytest.raises(RuntimeError, match="GPU"):
        indexer_topk(torch.randn(1, 4, 2, 8), torch.randn(1, 4, 2, 8), torch.rand(1, 4, 2), 2)
    with pytest.raises(RuntimeError, match="GPU"):
        page_select_hip(q, *alloc_page_meta(1, 2, 2, 64, torch.float32, "cpu"), 16, 1)
    with pytest.raises(ValueError):
        block_sparse_attention(q, k, k, ids, block_size=16, backend="triton")


def test_backend_report():
    """kernels/__init__.py:66-95: one backend, 'hip'."""
    assert backend_for() == "hip"
    with pytest.raises(ValueError):
        backend_for("torch")
    info = describe_backends()
    for key in ("platform", "torch", "hip_library", "gpu"):
        assert key in info


def test_page_meta_is_page_minor():
    mn, mx = alloc_page_meta(2, 3, 10, 64, torch.bfloat16, "cpu")
    assert mn.shape == (2, 3, 10, 64) and mn.stride(2) == 1 and mn.stride(3) == 12


def test_head_selection_refuses_what_its_grid_cannot_hold():
    """Before any launch: one row a workgroup (more than 256 pages) or four, fewer than
    2^32 threads."""
    import ctypes

    from linattn_amd import _native as N
    for rows, pages in ((1 << 26, 64), (1 << 24, 257)):
        a = N.LaQuestSelectArgs()
        a.q = a.page_min = a.page_max = a.out_idx = 4096  # (never read)
        a.B, a.Hq, a.Hkv, a.Tq, a.D = 1, 1, 1, rows, 64
        a.q_sb = a.q_sh = a.q_st = 64
        a.n_pages, a.page_size, a.k, a.pos_offset = pages, 16, 4, 0
        a.m_sb, a.m_sh, a.m_sp, a.m_sd = 64 * pages, 64 * pages, 1, pages
        a.q_dtype = a.meta_dtype = N.LA_F32
        assert N.load().la_quest_select_heads(ctypes.byref(a), None) == N.LA_ERR_UNSUPPORTED


@pytest.mark.parametrize("rows,pages,k,D,G,one", [
    (8, 256, 128, 64, 1, True), (8, 256, 129, 64, 1, False),        # the k^2 ranking
    (2047, 256, 65, 128, 1, False), (2048, 256, 65, 128, 1, True),
    (512, 512, 32, 128, 1, True), (513, 512, 32, 128, 1, False),    # the bounds read per row
    (257, 513, 32, 128, 1, False), (512, 1024, 32, 128, 4, True), (513, 257, 4, 64, 4, False),
    (1 << 20, 1024, 4, 64, 1, True), (8, 1025, 4, 64, 1, False),
])
def test_head_selection_takes_the_faster_form(rows, pages, k, D, G, one):
    from linattn_amd.kernels.quest_pages import _heads_in_one_kernel
    assert _heads_in_one_kernel(rows, pages, k, D, G) is one


@pytest.mark.parametrize("tq,tiled", [(8192, True), (32768, False)])
def test_list_tiles_bound_their_workspace(tq, tiled):
    """Tiles of many queries over a long cache, whose block lists grow with both: within
    512 MiB, or the row kernels (which need no workspace for so many rows)."""
    import ctypes

    from linattn_amd import _native as N
    a, kv = N.LaSparseAttnArgs(), N.LaKV()
    B, H, T, D = 64, 8, 262144, 128
    a.q, a.out, a.ids = 1 << 40, 1 << 44, 1 << 46  # (never read)
    a.B, a.Hq, a.Hkv, a.Tq, a.D = B, H, H, tq, D
    a.q_sb = a.o_sb = H * tq * D
    a.q_sh = a.o_sh = tq * D
    a.q_st = a.o_st = D
    a.ids_heads, a.ids_rows, a.N, a.unit = H, tq, 512, 64
    a.id_sb = a.id_sh = 0
    a.id_st, a.scale, a.q_dtype, a.out_dtype = 512, 0.1, N.LA_BF16, N.LA_BF16
    kv.k, kv.v, kv.T, kv.dtype = 1 << 47, 1 << 48, T, N.LA_BF16
    kv.k_sb = kv.v_sb = H * T * D
    kv.k_sh = kv.v_sh = T * D
    kv.k_st = kv.v_st = D
    n = N.load().la_sparse_attention_workspace(ctypes.byref(a), ctypes.byref(kv))
    assert (256 << 20) < n <= (512 << 20) if tiled else n == 0
