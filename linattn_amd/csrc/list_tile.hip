// Attention of many queries over per-query lists as tiles of 128 rows on the
// gfx950 matrix cores.
//
// The row kernels of sparse_attn.hip read every listed key once per query: a
// prefill whose queries carry their own lists (MoBA and Quest blocks, DSA
// tokens, sliding windows; variants/selection.py:86-116 builds the same
// masks) reads each K/V row hundreds of times.  Here a workgroup takes 128
// rows (the query heads of one KV head times consecutive queries), walks the
// 64-token key blocks that any of its rows lists, and multiplies each block
// against all of them on the matrix cores; what a row does not list is masked
// out of its softmax.
//
// Per call: list_mask_kernel turns the lists into bit masks (a bit per 64-token
// block when units are whole blocks, else a bit per token), stored block-major
// so that a tile reads its rows' bits side by side, and marks rows that list a
// unit twice (such a unit counts twice, which a bit cannot say).
// list_union_kernel writes each tile's block list, and leaves tiles whose rows
// share so little that reading each row's own keys is cheaper to the row
// kernel.  In a matrix product an infinity or a NaN of a block reaches rows that
// do not list it (0 * inf), but always as a result that is not finite: such rows
// are marked after the fact and done again by the row kernel, like the others
// left out (ListTileGate), which reads nothing that a row does not list.
//
// Tile kernel: four waves of 32 rows.  K and V blocks go global -> LDS by
// LDS-DMA, double buffered, one barrier per block.  S^T = K Q^T by
// v_mfma_f32_32x32x16_bf16 (A = K rows, B = Q held in registers) leaves a lane
// 16 scores of one query, so masks, maxima and sums are per lane; O^T = V^T P^T
// takes P from the same registers (the contraction index is mapped to the
// keys a lane holds) and V^T by LDS transpose reads.  The weights stay fp32:
// each is the exact sum of three bf16 terms (8 significant bits each), one
// product per term, so the result is the fp32 one (V and q, k are bf16 already).
#include <algorithm>
#include <numeric>

#include "kv_access.h"
#include "list_tile.h"

namespace la {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

constexpr int LT_M = 128, LT_NT = 256, LT_NW = 4, LT_D = 128, LT_BS = 64;
constexpr int LT_BLK = LT_BS * LT_D;   // elements of a staged K or V block
constexpr int LT_MAXB = 4096;          // key blocks of a cache (list positions in LDS)
// Tiles are left where that is clearly cheaper: both costs are good to a fifth, and
// left rows start when the tiles have ended.  Up to LT_ONE tiles are left together:
// they run at the same time, and as long as any of them when others are left (1024
// queries of 16 heads, 128 tokens of 8192 a row: 147 us in tiles, 137 in rows, 197 with
// half of the tiles left).
constexpr float LT_LEAVE = 1.25f;
constexpr int64_t LT_ONE = 4096;
enum { LT_TILES, LT_EACH, LT_TOGETHER };  // who decides: nobody, each tile, all of them

// Chunk swizzles of staged row r (16-byte chunks, 16 per row).  K: the 8-lane
// groups a ds_read_b128 pass serves together ({0,3}, {1,2}, ...) hold rows 8i..8i+7
// and 8j..8j+7 with bit 4 different, so these take even and odd chunks.  V: a
// transpose read's 32 lanes take 4 rows x 4 consecutive chunks.
__device__ __forceinline__ int lt_swz_k(int r) { return (2 * (r & 7)) ^ ((r >> 4) & 1); }
__device__ __forceinline__ int lt_swz_v(int r) { return 4 * (r & 3); }

struct LmKP {
  const int32_t *ids, *counts;
  uint32_t *mask;
  uint8_t *dup;
  int64_t id_sb, id_sh, id_st, N, unit, T;
  int64_t ids_heads, ids_rows, mheads, mrows;
  int32_t nblk, token, rw, lw;  // rw: mask rows per workgroup, lw: LDS words per row
  unsigned long long *balance;  // (set to 0 for list_union_kernel)
};

__global__ __launch_bounds__(256) void list_mask_kernel(LmKP p) {
  extern __shared__ __align__(16) uint32_t lbits[];
  __shared__ uint32_t s_dup[32];
  const int tid = threadIdx.x;
  const int64_t row0 = (int64_t)blockIdx.x * p.rw;
  for (int i = tid; i < p.rw * p.lw; i += 256) lbits[i] = 0u;
  if (tid < 32) s_dup[tid] = 0u;
  if (blockIdx.x == 0 && tid == 0) *p.balance = 0ull;
  __syncthreads();
  const int tpr = 256 / p.rw;  // threads of a row
  const int rl = tid / tpr, tl = tid % tpr;
  const int64_t m = row0 + rl;
  if (m < p.mrows) {
    const int64_t lrow = m % p.ids_rows;
    const int64_t ih = (m / p.ids_rows) % p.mheads, b = m / (p.ids_rows * p.mheads);
    const int32_t *list = p.ids + b * p.id_sb + ih * p.id_sh + lrow * p.id_st;
    int64_t n = p.N;
    if (p.counts) n = min(n, (int64_t)p.counts[(b * p.ids_heads + ih) * p.ids_rows + lrow]);
    uint32_t *bits = lbits + rl * p.lw;
    bool twice = false;
    constexpr int NB = 8;  // entries of a thread read before they are used
    for (int64_t e0 = tl; e0 < n; e0 += NB * tpr) {
      int32_t idb[NB];
#pragma unroll
      for (int x = 0; x < NB; ++x) idb[x] = e0 + x * tpr < n ? list[e0 + x * tpr] : -1;
#pragma unroll
      for (int x = 0; x < NB; ++x) {
        const int64_t id = idb[x];
        if (id < 0 || id * p.unit >= p.T) continue;
        if (p.token) {
          int64_t t0 = id * p.unit;
          const int64_t t1 = min(t0 + p.unit, p.T);
          while (t0 < t1) {  // the unit's tokens, word by word
            const int64_t te = min(t1, (t0 | 31) + 1);
            const uint32_t w = (0xffffffffu >> (32 - (int)(te - t0))) << (t0 & 31);
            twice |= (atomicOr(&bits[t0 >> 5], w) & w) != 0;
            t0 = te;
          }
        } else {
          const int64_t per = p.unit / LT_BS;
          for (int64_t kb = id * per; kb < min(id * per + per, (int64_t)p.nblk); ++kb) {
            const uint32_t w = 1u << (kb & 31);
            twice |= (atomicOr(&bits[kb >> 5], w) & w) != 0;
          }
        }
      }
    }
    if (twice) s_dup[rl] = 1u;
  }
  __syncthreads();
  const int nr = (int)min((int64_t)p.rw, p.mrows - row0);
  if (p.token) {
    uint2 *out = (uint2 *)p.mask;
    for (int i = tid; i < p.nblk * p.rw; i += 256) {
      const int r = i % p.rw, kb = i / p.rw;
      if (r < nr) out[(int64_t)kb * p.mrows + row0 + r] = *(const uint2 *)&lbits[r * p.lw + 2 * kb];
    }
  } else {
    const int nw = (p.nblk + 31) / 32;
    for (int i = tid; i < nw * p.rw; i += 256) {
      const int r = i % p.rw, x = i / p.rw;
      if (r < nr) p.mask[(int64_t)x * p.mrows + row0 + r] = lbits[r * p.lw + x];
    }
  }
  if (tid < nr) p.dup[row0 + tid] = (uint8_t)s_dup[tid];
}

struct LtKP {
  const uint16_t *q, *k, *v;
  void *out;
  const uint32_t *mask;
  const uint8_t *dup;
  uint16_t *list;   // [tile][nblk]: the blocks its rows list, ascending
  int32_t *nlist;   // [tile]: how many; -1: the tile is left to the row kernel
  // LT_TOGETHER: what walking costs more than the rows, summed over the tiles (two's
  // complement), which decides for all of them; else null
  unsigned long long *balance;
  uint8_t *rgate;   // [b][h][t]: a row whose result is not finite
  const int32_t *kv_len, *counts;
  float *ws_ml, *ws_acc;
  int64_t q_sb, q_sh, q_st, o_sb, o_sh, o_st;
  int64_t k_sb, k_sh, k_st, v_sb, v_sh, v_st;
  int64_t mrows, m_sb, m_sh, m_st, T, offset;
  int32_t Hq, Hkv, Tq, G, gt, qt, ntile, ngrp, nblk, splits, per_head, causal, out_dt, vec_out;
  int32_t ids_heads, nstream, N, unit, decide;
  float qscale, thr_gap, row_fixed, row_tok;  // row_*: see list_union_kernel
};

// Last key any query of the tile [t0, tl] may read, and its blocks.
__device__ __forceinline__ int lt_blocks(const LtKP &p, int64_t len, int tl) {
  const int64_t lim = p.causal ? min(len - 1, p.offset + tl) : len - 1;
  return lim < 0 ? 0 : (int)(lim / LT_BS) + 1;
}

// One workgroup per tile: the blocks any of its rows lists, within reach.
// The tile is left to the row kernel (count -1) when walking them for all 128 rows
// costs more than the lists row by row, entry by entry as that kernel walks them
// (to their counts, -1 entries too), by LT_LEAVE, in units of a row and token of a
// walked block (a shared list is read once for its heads there); or when every row
// lists a unit twice.
template <bool TOKEN>
__global__ __launch_bounds__(LT_NT) void list_union_kernel(LtKP p) {
  __shared__ uint32_t s_union[LT_MAXB / 32];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t tg = blockIdx.x;  // (b, group, tile)
  const int tile = (int)(tg % p.ntile), grp = (int)((tg / p.ntile) % p.ngrp);
  const int64_t b = tg / ((int64_t)p.ntile * p.ngrp);
  const int h0 = grp * p.gt;
  const int t0 = tile * p.qt, tl = min(t0 + p.qt, p.Tq) - 1;
  const int64_t len = p.kv_len ? min((int64_t)p.kv_len[b], p.T) : p.T;
  const int nb = lt_blocks(p, len, tl);
  const int64_t mbase = b * p.m_sb + (int64_t)(p.per_head ? h0 : h0 / p.G) * p.m_sh;
  const int heads = p.per_head ? p.gt : 1, nq = tl - t0 + 1;
  const int nr = p.m_st == 0 ? heads : heads * nq;  // mask rows of the tile (at most 128)
  // this lane's mask rows i and i + 64
  int64_t mr[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int i = min(lane + 64 * x, nr - 1);
    mr[x] = p.m_st == 0 ? mbase + i * p.m_sh : mbase + (int64_t)(i / nq) * p.m_sh + t0 + i % nq;
  }
  const bool in0 = lane < nr, in1 = lane + 64 < nr;
  // their list entries (with counts, mask rows are numbered as those are)
  int32_t ne[2] = {in0 ? p.N : 0, in1 ? p.N : 0};
  bool once = false;  // one of them lists no unit twice
  if (w == 0) {
    once = (in0 && p.dup[mr[0]] == 0) || (in1 && p.dup[mr[1]] == 0);
    if (p.decide != LT_TILES && p.counts) {
      if (in0) ne[0] = min(ne[0], max(p.counts[mr[0]], 0));
      if (in1) ne[1] = min(ne[1], max(p.counts[mr[1]], 0));
    }
  }
  for (int x = w; x * 32 < nb; x += LT_NW) {
    uint32_t word = 0;
    if constexpr (TOKEN) {
      const uint2 *mk = (const uint2 *)p.mask;
      const int kbe = min(32, nb - 32 * x);
      for (int k0 = 0; k0 < kbe; k0 += 8) {
        uint2 v[8], u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t at = (int64_t)(32 * x + min(k0 + e, kbe - 1)) * p.mrows;
          v[e] = in0 ? mk[at + mr[0]] : uint2{0, 0};
          u[e] = in1 ? mk[at + mr[1]] : uint2{0, 0};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (k0 + e >= kbe) break;
          if (__ballot((v[e].x | v[e].y | u[e].x | u[e].y) != 0) != 0) word |= 1u << (k0 + e);
        }
      }
    } else {
      const uint32_t in_nb = nb - 32 * x >= 32 ? 0xffffffffu : (1u << (nb - 32 * x)) - 1u;
      const uint32_t y = in0 ? p.mask[(int64_t)x * p.mrows + mr[0]] & in_nb : 0u;
      const uint32_t z = in1 ? p.mask[(int64_t)x * p.mrows + mr[1]] & in_nb : 0u;
      word = y | z;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) word |= (uint32_t)__shfl_xor((int)word, o, 64);
    }
    if (lane == 0) s_union[x] = word;
  }
  __syncthreads();
  if (w != 0) return;
  constexpr int WPL = LT_MAXB / 32 / 64;
  uint32_t bits[WPL], cnt = 0;
#pragma unroll
  for (int j = 0; j < WPL; ++j) {
    const int x = lane * WPL + j;
    bits[j] = x * 32 < nb ? s_union[x] : 0u;
    cnt += __popc(bits[j]);
  }
  uint32_t incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, o, 64);
    if (lane >= o) incl += y;
  }
  const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);
  bool rows = __ballot(once) == 0;  // (every row would be done again)
  if (p.decide != LT_TILES && !rows) {
    float entries = (float)ne[0] + (float)ne[1];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) entries += __shfl_xor(entries, o, 64);
    const float row_work = (p.row_fixed * (float)nr + p.row_tok * entries * (float)p.unit) *
                           (p.m_st == 0 ? (float)nq : 1.f);
    const float over = (float)total * (float)(LT_M * LT_BS) - LT_LEAVE * row_work;
    rows = p.decide == LT_EACH && over > 0.f;
    if (p.decide == LT_TOGETHER && lane == 0) atomicAdd(p.balance, (unsigned long long)(long long)over);
  }
  if (lane == 0) p.nlist[tg] = rows ? -1 : (int32_t)total;
  if (rows) return;
  uint16_t *out = p.list + tg * p.nblk;
  uint32_t at = incl - cnt;
#pragma unroll
  for (int j = 0; j < WPL; ++j) {
    uint32_t x = bits[j];
    while (x) {
      out[at++] = (uint16_t)((lane * WPL + j) * 32 + __ffs(x) - 1);
      x &= x - 1;
    }
  }
}

template <bool TOKEN>
__global__ __launch_bounds__(LT_NT, 2) void list_tile_kernel(LtKP p) {
  __shared__ __align__(16) uint16_t smem[4 * LT_BLK];  // K slots 0, 1, then V slots 0, 1
  __shared__ uint16_t s_list[LT_MAXB];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const int hf = lane >> 5, r32 = lane & 31;
  // Streams (b, head group, split) of tiles: the tiles of a stream run on one
  // XCD (its L2 keeps the stream's K/V), the longest causal rows first.
  uint32_t stream, tix;
  {
    const uint32_t wg = blockIdx.x, ns = (uint32_t)p.nstream, nt = (uint32_t)p.ntile;
    if (ns % 8 == 0) {
      stream = (wg & 7) + 8 * ((wg >> 3) / nt);
      tix = (wg >> 3) % nt;
    } else {
      stream = wg % ns;
      tix = wg / ns;
    }
  }
  const int tile = p.ntile - 1 - (int)tix;
  const int split = (int)(stream % (uint32_t)p.splits);
  const int grp = (int)((stream / (uint32_t)p.splits) % (uint32_t)p.ngrp);
  const int64_t b = stream / (uint32_t)(p.splits * p.ngrp);
  const int h0 = grp * p.gt, kvh = h0 / p.G;
  const int t0 = tile * p.qt;
  const int64_t len = p.kv_len ? min((int64_t)p.kv_len[b], p.T) : p.T;
  const int64_t mbase = b * p.m_sb + (int64_t)(p.per_head ? h0 : h0 / p.G) * p.m_sh;
  const int64_t tg = (b * p.ngrp + grp) * p.ntile + tile;
  const int nall = p.nlist[tg];
  if (nall < 0 || (p.balance && (long long)*p.balance > 0)) return;  // left to the row kernel
  const int e0 = (int)((int64_t)nall * split / p.splits);
  const int n = (int)((int64_t)nall * (split + 1) / p.splits) - e0;
  for (int i = tid; i < n; i += LT_NT) s_list[i] = p.list[tg * p.nblk + e0 + i];

  // q of this lane's row (B operand: dims 16 s + 8 hf .. + 7)
  const int row = 32 * w + r32, g = row / p.qt, t = t0 + row % p.qt;
  const bool live = t < p.Tq;
  const int h = h0 + g;
  bf16x8 qf[8];
  {
    const uint16_t *qp = p.q + b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)min(t, p.Tq - 1) * p.q_st + 8 * hf;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const bf16x8 *)(qp + 16 * s);
  }
  __syncthreads();

  const float NEG_INF = __int_as_float(0xff800000);
  float m = NEG_INF, thr = NEG_INF, l = 0.f, nmu = 0.f;
  f32x16 acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  const int64_t lim_r = live ? (p.causal ? min(len - 1, p.offset + t) : len - 1) : -1;
  const int lim32 = (int)max(lim_r, (int64_t)-1);
  const int64_t mr = p.m_st == 0 ? mbase + (p.per_head ? g : 0) * p.m_sh
                                 : mbase + (int64_t)(p.per_head ? g : 0) * p.m_sh + min(t, p.Tq - 1);
  const uint16_t *kbh = p.k + b * p.k_sb + kvh * p.k_sh, *vbh = p.v + b * p.v_sb + kvh * p.v_sh;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t *)smem);
  // LDS-DMA: instruction x of wave w fills rows 16 x + 4 w + lane / 16
  const int drow = 4 * w + (lane >> 4);
  uint32_t ko[4], vo[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int rr = 16 * x + drow;
    ko[x] = (uint32_t)((rr * p.k_st + 8 * ((lane & 15) ^ lt_swz_k(rr))) * 2);
    vo[x] = (uint32_t)((rr * p.v_st + 8 * ((lane & 15) ^ lt_swz_v(rr))) * 2);
  }
  auto dma = [&](const uint16_t *bh, int64_t st, const uint32_t (&off)[4], int kb, uint32_t slot, bool is_k) {
    const uint32_t m0 = lds0 + 2 * (slot * LT_BLK + 4 * wu * LT_D);
    if ((int64_t)(kb + 1) * LT_BS <= len) {
      const uint16_t *base = bh + (int64_t)kb * LT_BS * st;
#pragma unroll
      for (int x = 0; x < 4; ++x)
        asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(off[x]), "s"(base),
                     "{m0}"(m0 + 2 * 16 * x * LT_D) : "memory");
    } else {  // the last block: rows past the end read the last row (masked)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int rr = 16 * x + drow;
        const int64_t key = min((int64_t)kb * LT_BS + rr, len - 1);
        const int sw = is_k ? lt_swz_k(rr) : lt_swz_v(rr);
        asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(bh + key * st + 8 * ((lane & 15) ^ sw)),
                     "{m0}"(m0 + 2 * 16 * x * LT_D) : "memory");
      }
    }
  };
  // this lane's 64 mask bits of block kb, causality included
  auto load_mask = [&](int kb) -> uint2 {
    if constexpr (TOKEN) {
      return ((const uint2 *)p.mask)[(int64_t)kb * p.mrows + mr];
    } else {
      const uint32_t y = p.mask[(int64_t)(kb >> 5) * p.mrows + mr];
      return uint2{y, 0u};
    }
  };
  auto mask_bits = [&](uint2 raw, int kb) -> uint2 {
    if constexpr (!TOKEN) {
      const uint32_t f = (uint32_t)((int32_t)(raw.x << (31 - (kb & 31))) >> 31);
      raw = uint2{f, f};
    }
    const int d = lim32 - kb * LT_BS;  // last token of the block this row may read
    if (d < 63) {
      const uint64_t c = d < 0 ? 0ull : (2ull << d) - 1ull;
      raw.x &= (uint32_t)c;
      raw.y &= (uint32_t)(c >> 32);
    }
    return raw;
  };

  int kb = 0, kb_next = 0;
  uint2 mw{0, 0}, mw_next{0, 0};
  if (n > 0) {
    kb_next = __builtin_amdgcn_readfirstlane((int)s_list[0]);
    mw_next = load_mask(kb_next);
    dma(kbh, p.k_st, ko, kb_next, 0, true);
    dma(vbh, p.v_st, vo, kb_next, 2, false);
  }
  for (int j = 0; j < n; ++j) {
    const int par = j & 1;
    kb = kb_next;
    mw = mw_next;
    wait_vmcnt<0>();
    settle(mw.x);
    settle(mw.y);
    lds_barrier();  // block j has landed for every wave, block j - 1 is read
    if (j + 1 < n) {
      kb_next = __builtin_amdgcn_readfirstlane((int)s_list[j + 1]);
      mw_next = load_mask(kb_next);
      dma(kbh, p.k_st, ko, kb_next, par ^ 1, true);
      dma(vbh, p.v_st, vo, kb_next, 2 + (par ^ 1), false);
    }
    const uint2 bits = mask_bits(mw, kb);
    const bool none = (bits.x | bits.y) == 0u, all = (bits.x & bits.y) == 0xffffffffu;
    if (__ballot(!none) == 0) continue;  // no row of this wave lists the block
    const bool plain = __ballot(!none && !all) == 0;
    const uint16_t *sk = smem + par * LT_BLK, *sv = smem + (2 + par) * LT_BLK;
    f32x16 st[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) st[kt][i] = 0.f;
      const int kr = 32 * kt + r32, sw = lt_swz_k(kr);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const bf16x8 a = *(const bf16x8 *)&sk[kr * LT_D + 8 * ((2 * s + hf) ^ sw)];
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[s], st[kt], 0, 0, 0);
      }
    }
    // register i of a tile holds key 8 (i / 4) + 4 hf + i % 4
    if (!plain) {
      const uint32_t b0 = bits.x >> (4 * hf), b1 = bits.y >> (4 * hf);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int pos = 8 * (i >> 2) + (i & 3);
        st[0][i] = (b0 >> pos) & 1u ? st[0][i] : NEG_INF;
        st[1][i] = (b1 >> pos) & 1u ? st[1][i] : NEG_INF;
      }
    }
    float mx = st[0][0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, st[0][i]);
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[1][i]);
    if (none) mx = NEG_INF;
    // the reference maximum is raised only past 2^8 of headroom (the weights
    // stay below 256); both halves of a query keep the same one
    if (__ballot(mx > thr) != 0) {
      const float mn = fmaxf(m, pair32_max(mx));
      const float alpha = m == NEG_INF ? 0.f : fast_exp2((m - mn) * p.qscale);
      m = mn;
      thr = mn + p.thr_gap;
      nmu = mn == NEG_INF ? 0.f : -mn * p.qscale;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
    }
    // on a plain block a row outside it needs no select per score: 0 * s - inf
    // (NaN if s is not finite: the row is then done again)
    const bool skip = plain && none;
    const float qs = skip ? 0.f : p.qscale, nm = skip ? NEG_INF : nmu;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        st[kt][i] = fast_exp2(__builtin_fmaf(st[kt][i], qs, nm));
        l += st[kt][i];
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        // 8 weights as three bf16 terms each: the top halves of p, of what is
        // left, and of what is left of that (exact: 24 bits)
        uint32_t p1[4], p2[4], p3[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = st[kt][8 * ks + 2 * e], y = st[kt][8 * ks + 2 * e + 1];
          const uint32_t ux = __float_as_uint(x), uy = __float_as_uint(y);
          p1[e] = __builtin_amdgcn_perm(uy, ux, 0x07060302u);
          const float x2 = x - __uint_as_float(ux & 0xffff0000u), y2 = y - __uint_as_float(uy & 0xffff0000u);
          const uint32_t ux2 = __float_as_uint(x2), uy2 = __float_as_uint(y2);
          p2[e] = __builtin_amdgcn_perm(uy2, ux2, 0x07060302u);
          const float x3 = x2 - __uint_as_float(ux2 & 0xffff0000u), y3 = y2 - __uint_as_float(uy2 & 0xffff0000u);
          p3[e] = __builtin_amdgcn_perm(__float_as_uint(y3), __float_as_uint(x3), 0x07060302u);
        }
        const bf16x8 w1 = __builtin_bit_cast(bf16x8, u32x4{p1[0], p1[1], p1[2], p1[3]});
        const bf16x8 w2 = __builtin_bit_cast(bf16x8, u32x4{p2[0], p2[1], p2[2], p2[3]});
        const bf16x8 w3 = __builtin_bit_cast(bf16x8, u32x4{p3[0], p3[1], p3[2], p3[3]});
        // V^T: 16-lane group c of the wave points at rows k0 + i / 4 and reads
        // columns 32 dt + 16 (c % 2) + (its lane) of four keys
        const int vr = 32 * kt + 16 * ks + 4 * hf + ((lane & 15) >> 2);
        const int vc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), ve = 4 * (lane & 1);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          const int at = vr * LT_D + 8 * ((4 * dt + vc) ^ lt_swz_v(vr)) + ve;
          const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16 *)(sv + at));
          const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16 *)(sv + at + 8 * LT_D));
          const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w1, acc[dt], 0, 0, 0);
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w2, acc[dt], 0, 0, 0);
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w3, acc[dt], 0, 0, 0);
        }
      }
    }
  }
  l = pair32_sum(l);
  if (!live) return;
  // register i of dim tile dt holds dim 32 dt + 8 (i / 4) + 4 hf + i % 4
  if (p.splits > 1) {
    const int64_t Gl = p.per_head ? 1 : p.G, ih = p.per_head ? h : kvh, gl = p.per_head ? 0 : h % p.G;
    const int64_t pi = (((b * p.ids_heads + ih) * p.Tq + t) * Gl + gl) * p.splits + split;
    if (hf == 0) {
      p.ws_ml[2 * pi] = m == NEG_INF ? NEG_INF : m * p.qscale;
      p.ws_ml[2 * pi + 1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(float4 *)(p.ws_acc + pi * LT_D + 32 * dt + 8 * i + 4 * hf) =
            float4{acc[dt][4 * i], acc[dt][4 * i + 1], acc[dt][4 * i + 2], acc[dt][4 * i + 3]};
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bool fin = l < __int_as_float(0x7f800000);
  const int64_t o = b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)t * p.o_st + 4 * hf;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = l > 0.f ? acc[dt][4 * i + e] * inv : 0.f;
        fin = fin && fabsf(acc[dt][4 * i + e]) < __int_as_float(0x7f800000);
      }
      const int64_t at = o + 32 * dt + 8 * i;
      if (p.vec_out && p.out_dt == LA_BF16) {
        *(uint2 *)((uint16_t *)p.out + at) =
            uint2{(uint32_t)f32_to_bf16_bits(x[0]) | ((uint32_t)f32_to_bf16_bits(x[1]) << 16),
                  (uint32_t)f32_to_bf16_bits(x[2]) | ((uint32_t)f32_to_bf16_bits(x[3]) << 16)};
      } else if (p.vec_out && p.out_dt == LA_F32) {
        *(float4 *)((float *)p.out + at) = float4{x[0], x[1], x[2], x[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) store_from_f32(p.out, at + e, p.out_dt, x[e]);
      }
    }
  // the other half of the row's dims
  const uint64_t fm = __ballot(fin);
  if (hf == 0) p.rgate[(b * p.Hq + h) * p.Tq + t] = ((fm >> r32) & (fm >> (r32 + 32)) & 1) ? 0 : 1;
}

static size_t up256(size_t x) { return (x + 255) / 256 * 256; }

// Cost of a list row in the row kernels, in picoseconds of the whole device: of the
// row, and of each token of its list, by the heads that share it.  Fits of 64 to 2048
// tokens a row to a tenth (512 queries of 8 KV heads and 4096 keys, 2048 queries of 2
// or 8 and 16384 keys, units of 1, 8 and 64); over 65536 keys, which miss the L2s, 1.2
// (4 heads) to 1.7 (1 head) times as much a token.  (Four heads cost more a token than
// eight: held to four waves a SIMD their kernel spills 42 registers.)  Against
// LT_TILE_PS for a row and token of a walked block here (0.93-1.06 measured with
// every CU busy).  A row that its tile leaves costs LT_LEFT_PS more: its workgroup
// takes several one after another (16384 rows of one head and 32 tokens: 84 us in
// sparse_attn_mfma_kernel, 106 in sparse_attn_gated_kernel).
struct RowCost {
  float fixed, tok;
};
static RowCost row_ps(int64_t heads) {
  return heads == 8 ? RowCost{14000.f, 59.f} : heads == 4 ? RowCost{10000.f, 103.f}
         : heads == 2 ? RowCost{7000.f, 41.f} : RowCost{4000.f, 38.f};
}
constexpr float LT_TILE_PS = 1.1f, LT_LEFT_PS = 2000.f;
// The masks, the merge and the look for marked rows cost LT_EXTRA_US here, and four
// launches more on the host, so calls the row kernels finish sooner stay with them:
// those whose tokens take LT_MIN_ROW_US (512 listed tokens per query, 8 heads: 128
// queries 34 us by rows, 43 by tiles; 512 queries 93 and 50; 247 queries of 8 lists of
// 382 tokens for two heads, 3887 keys, 31 us of tokens: a DSA chunk 90 and 95; a window
// of 260 tokens over 511 keys, 8 heads, 30 us: the variant's prefill, which waits for
// its host, 126 and 138).  The host knows the width of lists, not their counts: wide lists
// that turn out nearly empty pay LT_EXTRA_US and the dearer rows (512 queries of 8
// lists over 8192 keys, units of 8: 1 unit a list 60 us by rows, 72 here, 4 units 62 and
// 94, 16 units 100 and 130; 64 units 247 and 154; 4 units and -1 to the full width,
// which the row kernel walks, 1418 and 116).
constexpr float LT_MIN_ROW_US = 38.f, LT_EXTRA_US = 20.f;
// Masks, block lists, marks and parts of one call (the row kernels need none of it).
constexpr size_t LT_MAX_BYTES = (size_t)512 << 20;

// Whether out may share memory with q: rows done again read q after their tile has
// stored (a row kernel reads a row of q before it writes that row of out).  Not where
// the spans of the two are apart, nor where rows lie in different places of what all
// strides are multiples of (halves of one tensor).
static bool out_in_q(const la_sparse_attn_args *a) {
  const int64_t eo = a->out_dtype == LA_F32 ? 4 : 2, nq = a->D * 2, no = a->D * eo;  // (q is bf16)
  const int64_t step[3][2] = {{a->q_sb * 2, a->o_sb * eo}, {a->q_sh * 2, a->o_sh * eo}, {a->q_st * 2, a->o_st * eo}};
  const int64_t count[3] = {a->B, a->Hq, a->Tq};
  int64_t g = 0, q0 = (int64_t)(uintptr_t)a->q, o0 = (int64_t)(uintptr_t)a->out;
  const int64_t d = o0 - q0;
  int64_t q1 = q0 + nq, o1 = o0 + no;
  for (int x = 0; x < 3; ++x) {
    if (count[x] == 1) continue;
    for (const int64_t s : {step[x][0], step[x][1]}) g = std::gcd(g, s);
    (step[x][0] < 0 ? q0 : q1) += (count[x] - 1) * step[x][0];
    (step[x][1] < 0 ? o0 : o1) += (count[x] - 1) * step[x][1];
  }
  if (o0 >= q1 || q0 >= o1) return false;
  if (g == 0) return true;
  const int64_t at = ((d % g) + g) % g;  // a row of out, past a row of q
  return !(at >= nq && g - at >= no);
}

ListTilePlan list_tile_plan(const la_sparse_attn_args *a, const la_kv *kv) {
  ListTilePlan pl;
  if (kv->page_table || kv->dtype != LA_BF16 || a->q_dtype != LA_BF16 || a->D != LT_D ||
      a->num_splits > 0 || !(a->scale > 0.f) || a->scale > 64.f)
    return pl;
  auto m8 = [](int64_t x) { return x % 8 == 0; };
  if (out_in_q(a)) return pl;
  if ((uintptr_t)a->q % 16 || !m8(a->q_sb) || !m8(a->q_sh) || !m8(a->q_st)) return pl;
  if (a->Tq < 32 || kv->T > (int64_t)LT_MAXB * LT_BS || a->offset < 0) return pl;
  const int64_t lim_st = (int64_t)1 << 23;  // 32-bit byte offsets of a block's rows
  if (kv->k_st < 0 || kv->v_st < 0 || kv->k_st >= lim_st || kv->v_st >= lim_st) return pl;
  const int64_t G = a->Hq / a->Hkv;
  const bool per_head = a->ids_heads == a->Hq;
  const bool pow2 = G == 1 || G == 2 || G == 4 || G == 8;
  if (!pow2 && !per_head) return pl;
  const int64_t reach = a->causal ? std::min(kv->T, a->offset + a->Tq) : kv->T;
  // Device time of the rows one by one, and of tiles that walk every block.
  const double o = a->causal ? (double)a->offset : (double)kv->T;
  auto mean = [&](double cap) {  // over the queries: keys within reach, at most cap
    const double n = (double)a->Tq, x = std::min(std::max(cap - o, 0.0), n);
    return (x * (o + (x + 1) / 2) + (n - x) * cap) / n;
  };
  const RowCost rc = row_ps(per_head ? 1 : G);
  const double n_rows = (double)(a->B * a->ids_heads * a->Tq);
  const double tok_ps = n_rows * rc.tok * mean((double)std::min(a->N * a->unit, kv->T));
  const double rows_ps = n_rows * rc.fixed + tok_ps;
  const int64_t gt = pow2 ? G : 1, qt = LT_M / gt;
  const double tile_ps = (double)(a->B * (a->Hq / gt) * ceil_div(a->Tq, qt) * LT_M) * LT_TILE_PS * mean((double)kv->T);
  if (tok_ps < LT_MIN_ROW_US * 1e6) return pl;
  // Surely cheaper: tiles.  Else whole-block lists, whose masks cost little,
  // are looked at tile by tile down to lists of 1/64 of what is within reach
  // (rows that share their blocks: 65536 keys, 17 blocks a row, 64 neighbours
  // drawing from the same 68 blocks: 269 us by rows, 109 by tiles).
  const bool sure = tile_ps + LT_EXTRA_US * 1e6 < rows_ps;
  if (!sure && (a->unit % LT_BS != 0 || reach > 64 * a->N * a->unit)) return pl;
  pl.sure = sure;
  pl.row_fixed = (rc.fixed + LT_LEFT_PS) / LT_TILE_PS;
  pl.row_tok = rc.tok / LT_TILE_PS;
  pl.gt = (int32_t)gt;
  pl.qt = (int32_t)qt;
  pl.ntile = (int32_t)ceil_div(a->Tq, pl.qt);
  pl.ngrp = (int32_t)(a->Hq / pl.gt);
  pl.nblk = (int32_t)ceil_div(kv->T, LT_BS);
  pl.token = a->unit % LT_BS != 0;
  // one mask for all that share a list (expanded lists have stride 0)
  const bool one_b = a->id_sb == 0 && !a->counts, one_h = a->id_sh == 0 && !a->counts;
  const int64_t mh = one_h ? 1 : a->ids_heads, mb = one_b ? 1 : a->B;
  pl.mrows = mb * mh * a->ids_rows;
  pl.m_st = a->ids_rows == 1 ? 0 : 1;
  pl.m_sh = one_h ? 0 : a->ids_rows;
  pl.m_sb = one_b ? 0 : mh * a->ids_rows;
  const int64_t tiles = a->B * pl.ngrp * pl.ntile;
  // Nothing to decide where even walking every block beats rows whose counts are 0 (or
  // whose lists, without counts, are walked to the end).
  const double least_ps = n_rows *
                          (rc.fixed + LT_LEFT_PS + (a->counts ? 0.0 : rc.tok * (double)(a->N * a->unit)));
  pl.decide = !sure ? LT_EACH : tile_ps < LT_LEAVE * least_ps ? LT_TILES
              : tiles <= LT_ONE ? LT_TOGETHER : LT_EACH;
  if (tiles > ((int64_t)1 << 24) || pl.mrows > ((int64_t)1 << 30)) return pl;
  // two workgroups per CU; parts of at least 8 blocks
  const int64_t want = ceil_div((int64_t)2 * num_cus(), tiles);
  pl.splits = (int32_t)std::max<int64_t>(1, std::min<int64_t>({want, ceil_div(reach, LT_BS) / 8, 16}));
  const size_t words = pl.token ? (size_t)pl.nblk * 2 : (size_t)ceil_div(pl.nblk, 32);
  if (pl.token && words * 4 > 49152) return pl;
  const size_t mask = words * 4 * (size_t)pl.mrows;
  size_t at = 0;
  auto take = [&](size_t n) { const size_t o = at; at += up256(n); return o; };
  pl.off_mask = take(mask);
  pl.off_dup = take((size_t)pl.mrows);
  pl.off_list = take((size_t)tiles * pl.nblk * 2);
  pl.off_nlist = take((size_t)tiles * 4);
  pl.off_balance = take(sizeof(uint64_t));
  pl.off_rgate = take((size_t)(a->B * a->Hq * a->Tq));
  if (pl.splits > 1) {
    const size_t parts = (size_t)(a->B * a->Hq * a->Tq) * pl.splits;
    pl.off_ml = take(parts * 2 * sizeof(float));
    pl.off_acc = take(parts * LT_D * sizeof(float));
  }
  if (at > LT_MAX_BYTES) return pl;
  pl.bytes = at;
  pl.use = true;
  return pl;
}

int list_tile_launch(const la_sparse_attn_args *a, const la_kv *kv, const ListTilePlan &pl,
                     void *ws, ListTileGate &gate, hipStream_t st) {
  uint8_t *base = (uint8_t *)ws;
  const bool per_head = a->ids_heads == a->Hq;
  LmKP m{};
  m.ids = a->ids;
  m.counts = a->counts;
  m.mask = (uint32_t *)(base + pl.off_mask);
  m.dup = base + pl.off_dup;
  m.id_sb = a->id_sb; m.id_sh = a->id_sh; m.id_st = a->id_st;
  m.N = a->N; m.unit = a->unit; m.T = kv->T;
  m.ids_heads = a->ids_heads; m.ids_rows = a->ids_rows;
  m.mheads = pl.m_sh == 0 ? 1 : a->ids_heads;
  m.mrows = pl.mrows;
  m.nblk = pl.nblk;
  m.token = pl.token;
  m.balance = (unsigned long long *)(base + pl.off_balance);
  m.lw = (int32_t)(pl.token ? 2 * pl.nblk : ceil_div(pl.nblk, 32));
  m.rw = 32;
  // rows share a workgroup (and write their masks side by side) as long as
  // there are workgroups for every CU
  while (m.rw > 1 && (m.rw * m.lw * 4 > 32768 || (pl.token && m.rw > 8) ||
                      ceil_div(pl.mrows, m.rw) < 2 * num_cus()))
    m.rw >>= 1;
  list_mask_kernel<<<dim3((unsigned)ceil_div(pl.mrows, m.rw)), 256, (size_t)m.rw * m.lw * 4, st>>>(m);
  LA_LAUNCHED();

  LtKP p{};
  p.q = (const uint16_t *)a->q;
  p.k = (const uint16_t *)kv->k;
  p.v = (const uint16_t *)kv->v;
  p.out = a->out;
  p.mask = m.mask;
  p.dup = m.dup;
  p.list = (uint16_t *)(base + pl.off_list);
  p.nlist = (int32_t *)(base + pl.off_nlist);
  p.decide = pl.decide;
  p.balance = pl.decide == LT_TOGETHER ? m.balance : nullptr;
  p.rgate = base + pl.off_rgate;
  p.kv_len = kv->kv_len;
  p.counts = a->counts;
  if (pl.splits > 1) {
    p.ws_ml = (float *)(base + pl.off_ml);
    p.ws_acc = (float *)(base + pl.off_acc);
  }
  p.q_sb = a->q_sb; p.q_sh = a->q_sh; p.q_st = a->q_st;
  p.o_sb = a->o_sb; p.o_sh = a->o_sh; p.o_st = a->o_st;
  p.k_sb = kv->k_sb; p.k_sh = kv->k_sh; p.k_st = kv->k_st;
  p.v_sb = kv->v_sb; p.v_sh = kv->v_sh; p.v_st = kv->v_st;
  p.mrows = pl.mrows; p.m_sb = pl.m_sb; p.m_sh = pl.m_sh; p.m_st = pl.m_st;
  p.T = kv->T;
  p.offset = a->offset;
  p.Hq = (int32_t)a->Hq; p.Hkv = (int32_t)a->Hkv; p.Tq = (int32_t)a->Tq;
  p.G = (int32_t)(a->Hq / a->Hkv);
  p.gt = pl.gt; p.qt = pl.qt; p.ntile = pl.ntile; p.ngrp = pl.ngrp; p.nblk = pl.nblk;
  p.splits = pl.splits;
  p.per_head = per_head;
  p.causal = a->causal;
  p.out_dt = a->out_dtype;
  const int64_t oal = a->out_dtype == LA_F32 ? 16 : 8;
  p.vec_out = (uintptr_t)a->out % oal == 0 && a->o_sb % 4 == 0 && a->o_sh % 4 == 0 && a->o_st % 4 == 0;
  p.ids_heads = (int32_t)a->ids_heads;
  p.N = (int32_t)a->N;
  p.unit = (int32_t)a->unit;
  p.nstream = (int32_t)(a->B * pl.ngrp * pl.splits);
  p.qscale = a->scale * 1.4426950408889634f;
  p.thr_gap = 8.f / p.qscale;
  p.row_fixed = pl.row_fixed;
  p.row_tok = pl.row_tok;
  const int64_t tiles = a->B * pl.ngrp * pl.ntile;
  const dim3 grid((unsigned)(tiles * pl.splits));
  if (pl.token) {
    list_union_kernel<true><<<dim3((unsigned)tiles), LT_NT, 0, st>>>(p);
    LA_LAUNCHED();
    list_tile_kernel<true><<<grid, LT_NT, 0, st>>>(p);
  } else {
    list_union_kernel<false><<<dim3((unsigned)tiles), LT_NT, 0, st>>>(p);
    LA_LAUNCHED();
    list_tile_kernel<false><<<grid, LT_NT, 0, st>>>(p);
  }
  LA_LAUNCHED();
  gate = ListTileGate{m.dup, p.rgate, p.nlist, p.balance, pl.m_sb, pl.m_sh, pl.m_st,
                      pl.qt, pl.ntile, pl.ngrp, pl.gt};
  return LA_OK;
}

}  // namespace la
