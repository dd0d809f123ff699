// Attention of many queries over per-query lists, as tiles on the matrix
// cores (see list_tile.hip).
#pragma once

#include "common.h"

namespace la {

// Sizes and workspace layout of one call; use == false: the row kernels run.
struct ListTilePlan {
  bool use = false;
  int32_t gt = 1;      // query heads of a tile (one KV head)
  int32_t qt = 0;      // queries of a tile: LT_M / gt
  int32_t ntile = 0;   // query tiles
  int32_t ngrp = 0;    // Hq / gt
  int32_t nblk = 0;    // 64-token key blocks
  int32_t splits = 1;  // parts a tile's block list is cut into
  bool token = false;  // masks hold a bit per token (else per 64-token block)
  int64_t mrows = 0, m_sb = 0, m_sh = 0, m_st = 0;  // mask rows and their strides over (b, list head, t)
  bool sure = false;   // full lists: tiles are surely cheaper
  int32_t decide = 0;  // which tiles are left (list_union_kernel)
  float row_fixed = 0.f, row_tok = 0.f;  // of a list row and of its tokens (list_union_kernel)
  size_t off_mask = 0, off_dup = 0, off_list = 0, off_nlist = 0, off_balance = 0, off_rgate = 0, off_ml = 0, off_acc = 0;
  size_t bytes = 0;
};

// Which rows the tiles left to the row kernel: row (b, list head, t) is
// attended there when it lists a unit twice (dup), when its tile was left out
// (nlist < 0, or all by the balance), or when a result of one of its query heads is not finite
// (rgate; written by the tile, or by the merge of its parts).
struct ListTileGate {
  const uint8_t *dup;
  uint8_t *rgate;        // [b][Hq][Tq]
  const int32_t *nlist;  // [b][ngrp][ntile]
  const unsigned long long *balance;  // null, or above 0 (signed): every tile
  int64_t m_sb, m_sh, m_st;
  int32_t qt, ntile, ngrp, gt;
  // (h and t below 2^31)
  __device__ __forceinline__ bool tile_left(int64_t b, int64_t h, int64_t t) const {
    return nlist[(b * ngrp + (uint32_t)h / (uint32_t)gt) * ntile + (uint32_t)t / (uint32_t)qt] < 0 ||
           (balance && (long long)*balance > 0);
  }
};

ListTilePlan list_tile_plan(const la_sparse_attn_args *a, const la_kv *kv);
// Masks, block lists and tiles.  The caller merges the parts (splits > 1: at
// ws + off_ml / off_acc) and then runs the rows left out.
int list_tile_launch(const la_sparse_attn_args *a, const la_kv *kv, const ListTilePlan &pl,
                     void *ws, ListTileGate &gate, hipStream_t st);

}  // namespace la
