// Block selection for block-sparse prefill (config C3), gfx950.
//
// The block-sparse estimator of MInferenceAttention._block_sparse
// (variants/selection.py:339-353): mean-pool q and k over 64-token blocks
// (block_reduce, core.py:102-120; the tail block repeats the last row), score
// every causal block pair with the pooled dot product, keep the top-k key
// blocks per (b, h, query block), then OR the sink blocks and the local window
// (which contains the diagonal block, selection.py:351).
//
// Arithmetic is fp64 and a fixed function of the inputs: pooled sums add rows
// in order and divide by the block size; block scores add fl(qbar_d*kbar_d)
// over d in order (never fused).  The positive 1/sqrt(D) factor of the
// reference does not change the ranking and is not applied.
#include <algorithm>

#include "common.h"
#include "topk.h"

namespace la {

// Rows of sequence b: lens[b] (clamped to [0, T]) in a ragged batch, else T.
__device__ __forceinline__ int64_t seq_rows(const int32_t *lens, int64_t b, int64_t T) {
  return lens ? min(max((int64_t)lens[b], (int64_t)0), T) : T;
}

// The block a pooling workgroup writes: blk0 + blockIdx.x, or, with per-
// sequence positions, the block of positions[b] (-1 when outside [0, nb)).
__device__ __forceinline__ int64_t pool_block(int64_t blk0, const int32_t *pos, int64_t b,
                                              int64_t bs, int64_t nb) {
  if (!pos) return blk0 + blockIdx.x;
  const int64_t p = pos[b];
  return (p >= 0 && p / bs < nb) ? p / bs : -1;
}

// qbar/kbar[b][h][blk][d] = (sum_{i<bs} x[b][h][min(blk*bs+i, T_b-1)][d]) / bs
// (T_b = seq_rows; a sequence without rows pools zeros, which no list reads)
__global__ __launch_bounds__(128) void mean_pool_kernel(const void *x, int dt, int64_t T, int64_t D,
                                                        int64_t sb, int64_t sh, int64_t st,
                                                        int64_t bs, int64_t H, int64_t nb,
                                                        double *out, const int32_t *lens,
                                                        int64_t blk0, const int32_t *pos) {
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int64_t blk = pool_block(blk0, pos, b, bs, nb);
  if (blk < 0) return;
  const int64_t base = b * sb + h * sh;
  T = seq_rows(lens, b, T);
  if (T == 0) {
    for (int64_t d = threadIdx.x; d < D; d += blockDim.x) out[((b * H + h) * nb + blk) * D + d] = 0.0;
    return;
  }
  for (int64_t d = threadIdx.x; d < D; d += blockDim.x) {
    double acc = 0.0;
    for (int64_t i = 0; i < bs; ++i) {
      const int64_t row = min(blk * bs + i, T - 1);
      acc = acc + load_as_f64(x, base + row * st + d, dt);
    }
    out[((b * H + h) * nb + blk) * D + d] = acc / (double)bs;
  }
}

// The same pooling with the block staged in LDS first: 16-byte loads, every
// row of the block in flight at once; thread d then adds the rows in order.
// Needs bs <= 64, D * element size a multiple of 16 bytes and <= 512 bytes,
// 16-byte aligned rows.
template <int ESZ, int NT>
__global__ __launch_bounds__(NT) void mean_pool_vec_kernel(const void *x, int dt, int64_t T,
                                                            int64_t D, int64_t sb, int64_t sh,
                                                            int64_t st, int64_t bs, int64_t H,
                                                            int64_t nb, double *out,
                                                            const int32_t *lens, int64_t blk0,
                                                            const int32_t *pos) {
  extern __shared__ __align__(16) unsigned char rows[];  // bs rows of D * ESZ bytes
  constexpr int CH = 64 * 512 / 16 / NT;                  // chunks per thread (max)
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int64_t blk = pool_block(blk0, pos, b, bs, nb);
  if (blk < 0) return;  // (workgroup-uniform)
  const int tid = threadIdx.x;
  T = seq_rows(lens, b, T);
  if (T == 0) {  // (workgroup-uniform)
    for (int64_t d = tid; d < D; d += NT) out[((b * H + h) * nb + blk) * D + d] = 0.0;
    return;
  }
  const int rb = (int)(D * ESZ);  // bytes per row
  const int cpr = rb / 16;
  const int total = (int)bs * cpr;
  const char *base = (const char *)x + (b * sb + h * sh) * ESZ;
  uint4 v[CH];
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int c = tid + u * NT;
    const int64_t row = min(blk * bs + c / cpr, T - 1);
    v[u] = c < total ? *(const uint4 *)(base + row * st * ESZ + (c % cpr) * 16) : uint4{0, 0, 0, 0};
  }
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int c = tid + u * NT;
    if (c < total) *(uint4 *)(rows + (c / cpr) * rb + (c % cpr) * 16) = v[u];
  }
  __syncthreads();
  for (int64_t d = tid; d < D; d += NT) {
    double acc = 0.0;
    for (int64_t i = 0; i < bs; ++i) {
      const unsigned char *e = rows + i * rb + d * ESZ;
      double xv;
      if constexpr (ESZ == 4) {
        xv = (double)*(const float *)e;
      } else {
        const uint32_t bits = *(const uint16_t *)e;
        xv = dt == LA_BF16 ? (double)bf16_bits_to_f32(bits)
                           : (double)__half2float(__ushort_as_half((uint16_t)bits));
      }
      acc = acc + xv;
    }
    out[((b * H + h) * nb + blk) * D + d] = acc / (double)bs;
  }
}

// scores[(b*Hq+h)*nq + i][j] = sum_d fl(q[b,h,i,d] * kbar[b,h/G,j,d]), fp64, d
// increasing, each product rounded before it is added.  Row i sits at position
// pos0 + i*qunit and column j starts at j*kunit: columns past every row of a
// group are skipped (causal: their scores are never read).
struct ScKP {
  const void *q;  // at element strides q_sb, q_sh, q_st, unit stride over d
  const double *kbar;
  double *scores;
  int64_t q_sb, q_sh, q_st;
  int64_t Hq, Hkv, nq, nkb, D, pos0, qunit, kunit;
  int32_t q_dt;
};

constexpr int SC_NC = 8, SC_D = 128;  // columns of a wave, most dims

template <int DT>
__device__ __forceinline__ double sc_widen(const uint4 &v, int i) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (DT == LA_F32)
    return (double)__uint_as_float(w[i]);
  else if constexpr (DT == LA_BF16)
    return (double)((i & 1) ? bf16hi(w[i / 2]) : bf16lo(w[i / 2]));
  else
    return (double)__half2float(__ushort_as_half((uint16_t)(w[i / 2] >> (16 * (i & 1)))));
}

// Many rows of q as stored (the gates): a lane is R rows; a workgroup takes 64 R
// rows and 4 SC_NC columns, SC_NC per wave.  The columns' means sit in LDS and
// are read as broadcasts; q is read in its own type, by the four waves together
// (widened ahead of time it cost a pass of its own: 27 us for 1024 queries of 32
// heads).  Bound by its fp64 instructions (a multiply and an add per product: they
// round separately) and the broadcasts that feed them.  The scores leave through
// LDS as runs of 4 SC_NC per row: written SC_NC at a time, at the power-of-two
// strides that rows have, they took longer than the products.  1024 queries of 32
// heads on 64 blocks, D = 128: 59 us with the widening pass and 4 x 4 scores per
// thread, 27 like this.  Rows of 8-byte values (pooled q) need four times as many
// scattered loads and stay with block_score_kernel (64 heads of 512 x 512, causal:
// 144 us there, 205-290 in forms of this one).
template <int DT, int R>
__global__ __launch_bounds__(256) void row_score_kernel(ScKP p) {
  constexpr int EV = DT == LA_F32 ? 4 : 8;  // values of a 16-byte load
  constexpr int ESZ = 16 / EV, NL = 8 / EV;
  constexpr int WC = 4 * SC_NC, LD = WC + 1, ROWS = 64 * R;
  extern __shared__ __align__(16) double lds[];  // WC columns of D means; then ROWS rows of LD scores
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t j0 = (int64_t)blockIdx.x * WC, i0 = (int64_t)blockIdx.y * ROWS;
  const int64_t bh = blockIdx.z, b = bh / p.Hq, h = bh % p.Hq;
  // columns that start past every row's position: never read
  const int64_t last = p.pos0 + min(i0 + ROWS - 1, p.nq - 1) * p.qunit;
  if (j0 * p.kunit > last) return;
  const int D = (int)p.D, nc = (int)min((int64_t)WC, p.nkb - j0);
  const double *kr = p.kbar + ((b * p.Hkv + h / (p.Hq / p.Hkv)) * p.nkb + j0) * D;
  for (int x = tid; x < WC * D; x += 256) lds[x] = x < nc * D ? kr[x] : 0.0;
  __syncthreads();
  double acc[R][SC_NC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < SC_NC; ++c) acc[r][c] = 0.0;
  if (SC_NC * w < nc && (j0 + SC_NC * w) * p.kunit <= last) {
    const double *sk = lds + SC_NC * w * D;
    const char *qr[R];
    uint4 nx[R][NL];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      qr[r] = (const char *)p.q + (b * p.q_sb + h * p.q_sh + min(i0 + 64 * r + lane, p.nq - 1) * p.q_st) * ESZ;
#pragma unroll
      for (int y = 0; y < NL; ++y) nx[r][y] = *(const uint4 *)(qr[r] + 16 * y);
    }
    for (int d0 = 0; d0 < D; d0 += 8) {
      double x[R][8];
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[r][e] = sc_widen<DT>(nx[r][e / EV], e % EV);
        if (d0 + 8 < D) {
#pragma unroll
          for (int y = 0; y < NL; ++y) nx[r][y] = *(const uint4 *)(qr[r] + (d0 + 8) * ESZ + 16 * y);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; e += 2)
#pragma unroll
        for (int c = 0; c < SC_NC; ++c) {
          const double2 k2 = *(const double2 *)&sk[c * D + d0 + e];
#pragma unroll
          for (int r = 0; r < R; ++r)
            acc[r][c] = add_product(add_product(acc[r][c], x[r][e], k2.x), x[r][e + 1], k2.y);
        }
    }
  }
  __syncthreads();  // the means are read
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < SC_NC; ++c) lds[(64 * r + lane) * LD + SC_NC * w + c] = acc[r][c];
  __syncthreads();
  const int nr = (int)min((int64_t)ROWS, p.nq - i0);
  double *out = p.scores + (bh * p.nq + i0) * p.nkb + j0;
  for (int x = tid; x < nr * WC; x += 256) {
    const int i = x / WC, c = x % WC;
    if (c < nc) out[i * p.nkb + c] = lds[i * LD + c];
  }
}

// Few rows (decode): the heads of a KV head and their rows (at most SF_ROWS
// together) against 64 columns; the columns' means, read once for all of
// them, land in LDS in one memory round trip.  Bound by that read.
constexpr int SF_ROWS = 8, SF_D = 128;
__global__ __launch_bounds__(256) void few_row_score_kernel(ScKP p) {
  __shared__ double sk[64][SF_D + 1];
  __shared__ __align__(16) double sq[SF_ROWS][SF_D];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t j0 = (int64_t)blockIdx.x * 64;
  const int64_t kvh = blockIdx.y, b = blockIdx.z, G = p.Hq / p.Hkv;
  if (j0 * p.kunit > p.pos0 + (p.nq - 1) * p.qunit) return;
  const int D = (int)p.D, nc = (int)min((int64_t)64, p.nkb - j0), rows = (int)(G * p.nq);
  const double *kr = p.kbar + ((b * p.Hkv + kvh) * p.nkb + j0) * D;
  constexpr int PER = 64 * SF_D / 2 / 256;
  const int total = nc * D / 2;
  double2 v[PER];
#pragma unroll
  for (int x = 0; x < PER; ++x)
    v[x] = tid + 256 * x < total ? ((const double2 *)kr)[tid + 256 * x] : double2{0.0, 0.0};
  for (int x = tid; x < rows * D; x += 256) {
    const int r = x / D, d = x % D;  // row r = (head g, row i)
    sq[r][d] = load_as_f64(p.q, b * p.q_sb + (kvh * G + r / p.nq) * p.q_sh + (r % p.nq) * p.q_st + d, p.q_dt);
  }
#pragma unroll
  for (int x = 0; x < PER; ++x) {
    const int at = 2 * (tid + 256 * x);
    if (at < 2 * total) {
      sk[at / D][at % D] = v[x].x;
      sk[at / D][at % D + 1] = v[x].y;
    }
  }
  __syncthreads();
  for (int r = w; r < rows; r += 4) {
    double acc = 0.0;
    for (int d = 0; d < D; ++d) acc = add_product(acc, sq[r][d], sk[lane][d]);
    if (lane < nc)
      p.scores[((b * p.Hq + kvh * G + r / p.nq) * p.nq + r % p.nq) * p.nkb + j0 + lane] = acc;
  }
}

// Any shape (and pooled q, F64): 4 x 4 scores per thread on 64 x 64 tiles staged
// in LDS.  VEC (pooled q and means in 16-byte pieces): the next 32 dims are in
// flight, all loads at once, while these are multiplied (loaded one by one between
// two barriers they took longer than the products).  Bound by the fp64 instructions
// (a multiply and an add per product) and as many LDS clocks.  64 heads of 512 x 512
// on 128 dims, causal: 203 us loaded one by one, 157 loaded ahead, 144 with columns
// read in runs of 256 bytes and whole slices unrolled (56 for the instructions; held
// to 128 registers for a fourth workgroup per CU it spills and takes 168).
// TQ = 4: one score per thread, for up to four rows a head, of which a 64-row tile
// would stage and multiply 60 empty ones.  Gate calls of 64 heads on 4 KV heads, one
// query, 256 blocks, batch 8: 61 us on 64-row tiles, 30 here; 16 heads, four queries,
// D = 192, batch 4: 34 and 20.
constexpr int BS_DC = 32, BS_NT = 256;
template <bool F64, bool VEC, int TQ = 64>
__global__ __launch_bounds__(BS_NT) void block_score_kernel(ScKP p) {
  constexpr int RQ = TQ == 64 ? 4 : 1, RK = RQ, TX = BS_NT / (TQ / RQ), TK = TX * RK;
  constexpr int NV = TQ * BS_DC / (2 * BS_NT);  // pairs of a thread's share of a slice
  static_assert(TK == 64 && (TQ == 64 || TQ == 4) && (!VEC || (F64 && TQ == TK)), "");
  __shared__ __align__(16) double sq[BS_DC][TQ + 2];
  __shared__ __align__(16) double sk[BS_DC][TK + 2];
  const int tid = threadIdx.x;
  // rows RQ*tq.., columns 2*tk, 2*tk + 1 and TK/2 on: 16 threads read 256 bytes in a row
  const int tq = tid / TX, tk = tid % TX;
  auto col = [&](int c) { return RK == 1 ? tk : (c >> 1) * (TK / 2) + 2 * tk + (c & 1); };
  const int64_t i0 = (int64_t)blockIdx.y * TQ, j0 = (int64_t)blockIdx.x * TK;
  const int64_t bh = blockIdx.z;
  const int64_t b = bh / p.Hq, h = bh % p.Hq;
  if (j0 * p.kunit > p.pos0 + min(i0 + TQ - 1, p.nq - 1) * p.qunit) return;  // all in the future
  const int64_t q0 = b * p.q_sb + h * p.q_sh;
  const double *kb = p.kbar + (b * p.Hkv + h / (p.Hq / p.Hkv)) * p.nkb * p.D;
  double acc[RQ][RK];
#pragma unroll
  for (int a = 0; a < RQ; ++a)
#pragma unroll
    for (int c = 0; c < RK; ++c) acc[a][c] = 0.0;
  double2 vq[VEC ? NV : 1], vk[VEC ? NV : 1];
  // (rows and dims past the end read the last ones; their sums are not stored or not formed)
  auto fetch = [&](int64_t d0) {
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      const int at = tid + BS_NT * x, r = at / (BS_DC / 2);
      const int64_t d = min(d0 + 2 * (at % (BS_DC / 2)), p.D - 2);
      vq[x] = *(const double2 *)((const double *)p.q + q0 + min(i0 + r, p.nq - 1) * p.q_st + d);
      vk[x] = *(const double2 *)(kb + min(j0 + r, p.nkb - 1) * p.D + d);
    }
  };
  if constexpr (VEC) fetch(0);
  for (int64_t d0 = 0; d0 < p.D; d0 += BS_DC) {
    const int dn = (int)min((int64_t)BS_DC, p.D - d0);
    __syncthreads();
    if constexpr (VEC) {
#pragma unroll
      for (int x = 0; x < NV; ++x) {
        const int at = tid + BS_NT * x, r = at / (BS_DC / 2), dd = 2 * (at % (BS_DC / 2));
        sq[dd][r] = vq[x].x;
        sq[dd + 1][r] = vq[x].y;
        sk[dd][r] = vk[x].x;
        sk[dd + 1][r] = vk[x].y;
      }
    } else {
      for (int x = tid; x < TQ * BS_DC; x += BS_NT) {
        const int r = x / BS_DC, dd = x % BS_DC;
        const int64_t at = q0 + (i0 + r) * p.q_st + d0 + dd;
        double v = 0.0;
        if (dd < dn && i0 + r < p.nq) v = F64 ? ((const double *)p.q)[at] : load_as_f64(p.q, at, p.q_dt);
        sq[dd][r] = v;
      }
      for (int x = tid; x < TK * BS_DC; x += BS_NT) {
        const int r = x / BS_DC, dd = x % BS_DC;
        sk[dd][r] = (dd < dn && j0 + r < p.nkb) ? kb[(j0 + r) * p.D + d0 + dd] : 0.0;
      }
    }
    __syncthreads();
    if constexpr (VEC)
      if (d0 + BS_DC < p.D) fetch(d0 + BS_DC);
    auto products = [&](int dd) {
      double qv[RQ], kv[RK];
#pragma unroll
      for (int a = 0; a < RQ; ++a) qv[a] = sq[dd][RQ * tq + a];
#pragma unroll
      for (int c = 0; c < RK; ++c) kv[c] = sk[dd][col(c)];
#pragma unroll
      for (int a = 0; a < RQ; ++a)
#pragma unroll
        for (int c = 0; c < RK; ++c) acc[a][c] = add_product(acc[a][c], qv[a], kv[c]);
    };
    if (dn == BS_DC) {
#pragma unroll 8
      for (int dd = 0; dd < BS_DC; ++dd) products(dd);
    } else {
      for (int dd = 0; dd < dn; ++dd) products(dd);
    }
  }
#pragma unroll
  for (int a = 0; a < RQ; ++a) {
    const int64_t i = i0 + RQ * tq + a;
    if (i >= p.nq) continue;
#pragma unroll
    for (int c = 0; c < RK; ++c) {
      const int64_t j = j0 + col(c);
      if (j < p.nkb) p.scores[(bh * p.nq + i) * p.nkb + j] = acc[a][c];
    }
  }
}

template <int DT>
static void launch_row_scores(const ScKP &p, int64_t B, hipStream_t st) {
  const int R = p.nq > 64 ? 2 : 1;
  const dim3 grid((unsigned)ceil_div(p.nkb, 4 * SC_NC), (unsigned)ceil_div(p.nq, 64 * R), (unsigned)(B * p.Hq));
  const size_t lds = std::max<size_t>(4 * SC_NC * p.D, 64 * R * (4 * SC_NC + 1)) * sizeof(double);
  if (R == 2)
    row_score_kernel<DT, 2><<<grid, 256, lds, st>>>(p);
  else
    row_score_kernel<DT, 1><<<grid, 256, lds, st>>>(p);
}

// Scores of every row and column of (B * Hq) heads.  Up to SF_ROWS rows per KV
// head of up to SF_D dims take the decode form that reads the means once for all of
// them, other calls of up to four rows per head the 4-row tiles; the row form needs
// q rows in 16-byte pieces, and below 16 rows its lanes are mostly idle.
static void block_scores(const ScKP &p, int64_t B, hipStream_t st) {
  const int64_t ev = p.q_dt == LA_F32 ? 4 : 8;
  if (p.Hq / p.Hkv * p.nq <= SF_ROWS && p.D <= SF_D && p.D % 2 == 0 && (uintptr_t)p.kbar % 16 == 0) {
    few_row_score_kernel<<<dim3((unsigned)ceil_div(p.nkb, 64), (unsigned)p.Hkv, (unsigned)B), 256, 0, st>>>(p);
    return;
  }
  const dim3 tiles((unsigned)ceil_div(p.nkb, 64), (unsigned)ceil_div(p.nq, 64), (unsigned)(B * p.Hq));
  const bool rows = p.nq >= 16 && p.D % 8 == 0 && p.D <= SC_D && (uintptr_t)p.q % 16 == 0 &&
                    p.q_sb % ev == 0 && p.q_sh % ev == 0 && p.q_st % ev == 0;
  const bool vec = p.D % 2 == 0 && (uintptr_t)p.q % 16 == 0 && (uintptr_t)p.kbar % 16 == 0 &&
                   p.q_sb % 2 == 0 && p.q_sh % 2 == 0 && p.q_st % 2 == 0;
  const dim3 few(tiles.x, 1, tiles.z);
  if (p.nq <= 4 && p.q_dt == LA_F64)
    block_score_kernel<true, false, 4><<<few, BS_NT, 0, st>>>(p);
  else if (p.nq <= 4)
    block_score_kernel<false, false, 4><<<few, BS_NT, 0, st>>>(p);
  else if (p.q_dt == LA_F64 && vec)
    block_score_kernel<true, true><<<tiles, BS_NT, 0, st>>>(p);
  else if (p.q_dt == LA_F64)
    block_score_kernel<true, false><<<tiles, BS_NT, 0, st>>>(p);
  else if (!rows)
    block_score_kernel<false, false><<<tiles, BS_NT, 0, st>>>(p);
  else if (p.q_dt == LA_F32)
    launch_row_scores<LA_F32>(p, B, st);
  else if (p.q_dt == LA_BF16)
    launch_row_scores<LA_BF16>(p, B, st);
  else
    launch_row_scores<LA_F16>(p, B, st);
}

// Mean of every `bs` rows of x[b][h] (rows past T_b repeat row T_b-1) into
// out[b][h][blk][d] in fp64; bs = 1 is the exact widening to fp64.  T_b is
// lens[b] (ragged batch) or T.  Blocks blk0 .. blk0 + npool - 1 (all nb by
// default), or the block of pos[b] for each sequence b (npool = 1).
static void pool_rows(const void *x, int dt, int64_t B, int64_t H, int64_t T, int64_t D, int64_t sb,
                      int64_t sh, int64_t s_t, int64_t bs, int64_t nb, double *out,
                      hipStream_t st, const int32_t *lens = nullptr, int64_t blk0 = 0,
                      int64_t npool = -1, const int32_t *pos = nullptr) {
  const int64_t esz = dt == LA_F32 ? 4 : 2;
  if (npool < 0) npool = nb;
  const dim3 grid((unsigned)npool, (unsigned)H, (unsigned)B);
  const bool vec = bs <= 64 && (D * esz) % 16 == 0 && D * esz <= 512 && (uintptr_t)x % 16 == 0 &&
                   (sb * esz) % 16 == 0 && (sh * esz) % 16 == 0 && (s_t * esz) % 16 == 0;
  const size_t lds = (size_t)(bs * D * esz);
  // 128 threads when one thread per d covers the row (the block stays in LDS
  // only while it is summed, so several blocks per CU overlap)
  if (vec && esz == 4 && D <= 128)
    mean_pool_vec_kernel<4, 128><<<grid, 128, lds, st>>>(x, dt, T, D, sb, sh, s_t, bs, H, nb, out, lens, blk0, pos);
  else if (vec && esz == 4)
    mean_pool_vec_kernel<4, 256><<<grid, 256, lds, st>>>(x, dt, T, D, sb, sh, s_t, bs, H, nb, out, lens, blk0, pos);
  else if (vec && D <= 128)
    mean_pool_vec_kernel<2, 128><<<grid, 128, lds, st>>>(x, dt, T, D, sb, sh, s_t, bs, H, nb, out, lens, blk0, pos);
  else if (vec)
    mean_pool_vec_kernel<2, 256><<<grid, 256, lds, st>>>(x, dt, T, D, sb, sh, s_t, bs, H, nb, out, lens, blk0, pos);
  else
    mean_pool_kernel<<<grid, 128, 0, st>>>(x, dt, T, D, sb, sh, s_t, bs, H, nb, out, lens, blk0, pos);
}

struct BsLayout {
  int64_t nqb, nkb, qbar_off, kbar_off, sc_off, bytes;
};

static BsLayout layout(const la_block_select_args *a) {
  BsLayout L{};
  L.nqb = ceil_div(a->T, a->block);
  L.nkb = L.nqb;
  L.qbar_off = 0;
  L.kbar_off = L.qbar_off + a->B * a->Hq * L.nqb * a->D * 8;
  L.sc_off = L.kbar_off + a->B * a->Hkv * L.nkb * a->D * 8;
  L.bytes = L.sc_off + a->B * a->Hq * L.nqb * L.nkb * 8;
  return L;
}

static int validate(const la_block_select_args *a) {
  LA_REQUIRE(a && a->q && a->k && a->out_idx, "la_block_select: null pointer");
  LA_REQUIRE(a->B > 0 && a->Hq > 0 && a->Hkv > 0 && a->T > 0 && a->D > 0 && a->block > 0,
             "la_block_select: bad shape");
  LA_REQUIRE(a->Hq % a->Hkv == 0, "n_heads must be a multiple of n_kv_heads");
  LA_REQUIRE(a->topk >= 1 && a->sink_blocks >= 0 && a->window_blocks >= 0, "la_block_select: budget");
  LA_REQUIRE(a->width >= a->topk + a->sink_blocks + a->window_blocks,
             "la_block_select: width < topk + sink + window");
  LA_REQUIRE(a->in_dtype == LA_F32 || a->in_dtype == LA_BF16 || a->in_dtype == LA_F16,
             "la_block_select: q/k dtype");
  return LA_OK;
}

}  // namespace la

using namespace la;

extern "C" size_t la_block_select_workspace(const la_block_select_args *a) {
  if (validate(a) != LA_OK) return 0;
  return (size_t)layout(a).bytes;
}

extern "C" int la_block_select(const la_block_select_args *a, void *stream) {
  int rc = validate(a);
  if (rc != LA_OK) return rc;
  const BsLayout L = layout(a);
  if (!a->workspace || a->ws_bytes < L.bytes)
    return fail(LA_ERR_WORKSPACE, "la_block_select: workspace %lld < %lld bytes",
                (long long)a->ws_bytes, (long long)L.bytes);
  hipStream_t st = (hipStream_t)stream;
  char *ws = (char *)a->workspace;
  double *qbar = (double *)(ws + L.qbar_off);
  double *kbar = (double *)(ws + L.kbar_off);
  double *sc = (double *)(ws + L.sc_off);
  pool_rows(a->q, a->in_dtype, a->B, a->Hq, a->T, a->D, a->q_sb, a->q_sh, a->q_st, a->block, L.nqb,
            qbar, st, a->lengths);
  LA_LAUNCHED();
  pool_rows(a->k, a->in_dtype, a->B, a->Hkv, a->T, a->D, a->k_sb, a->k_sh, a->k_st, a->block, L.nkb,
            kbar, st, a->lengths);
  LA_LAUNCHED();
  ScKP sp{};
  sp.q = qbar;
  sp.q_dt = LA_F64;
  sp.q_st = a->D;
  sp.q_sh = L.nqb * a->D;
  sp.q_sb = a->Hq * L.nqb * a->D;
  sp.kbar = kbar;
  sp.scores = sc;
  sp.Hq = a->Hq;
  sp.Hkv = a->Hkv;
  sp.nq = L.nqb;
  sp.nkb = L.nkb;
  sp.D = a->D;
  sp.qunit = sp.kunit = 1;
  block_scores(sp, a->B, st);
  LA_LAUNCHED();
  TopkKParams tp{};
  tp.scores = sc;
  tp.row_stride = L.nkb;
  tp.G = 1;
  tp.Tq = L.nqb;
  tp.NG = a->B * a->Hq * L.nqb;
  tp.t_base = 0;
  tp.out_tq = L.nqb;
  tp.n = L.nkb;
  tp.k = a->topk;
  tp.width = a->width;
  tp.pos_off = 0;  // query block qb: key blocks kb <= qb, own block qb
  tp.pos_unit = 1;
  tp.sink = a->sink_blocks;
  tp.window = a->window_blocks;
  tp.order = 1;
  tp.out_idx = a->out_idx;
  tp.out_count = a->out_count;
  // ragged: the query blocks of sequence b at or past its length select nothing
  tp.b_lens = a->lengths;
  tp.rows_per_b = a->Hq * L.nqb;
  tp.b_len_unit = a->block;
  return topk_launch(tp, st);
}

// ------------------------------------------------------------ gate select --
// Per-query block routing: MoBA's gate (variants/selection.py:624-634) and
// the blockwise selection of NSA (variants/native_sparse.py:78-93), which
// compute the same thing: g[j] = q_t . mean(K block j) over the visible
// blocks (start <= pos_t = offset + t), the top-k blocks by gate, and the
// query's own block OR'd in.  The gates are fp64, fl(q_d * kbar_d) added
// over d in order, without the positive 1/sqrt(D) factor (it does not change
// the ranking); ties go to the lowest block.
namespace la {
struct GsLayout {
  int64_t nkb, kbar_off, sc_off, bytes;
};
static GsLayout gs_layout(const la_gate_select_args *a) {
  GsLayout L{};
  L.nkb = ceil_div(a->T, a->block);
  L.kbar_off = 0;
  // (no pooled keys when the caller keeps them)
  L.sc_off = L.kbar_off + (a->kbar ? 0 : a->B * a->Hkv * L.nkb * a->D * 8);
  L.bytes = L.sc_off + a->B * a->Hq * a->Tq * L.nkb * 8;
  return L;
}
static int gs_validate(const la_gate_select_args *a) {
  LA_REQUIRE(a && a->q && (a->k || a->kbar) && a->out_idx, "la_gate_select: null pointer");
  LA_REQUIRE(a->B > 0 && a->Hq > 0 && a->Hkv > 0 && a->Tq > 0 && a->T > 0 && a->D > 0 &&
                 a->block > 0,
             "la_gate_select: bad shape");
  LA_REQUIRE(a->Hq % a->Hkv == 0, "n_heads must be a multiple of n_kv_heads");
  LA_REQUIRE(a->topk >= 1, "la_gate_select: topk");
  LA_REQUIRE(a->offset >= 0, "la_gate_select: offset");
  LA_REQUIRE(a->width >= std::min(a->topk, ceil_div(a->T, a->block)) + 1,
             "la_gate_select: width < min(topk, blocks) + 1");
  LA_REQUIRE(a->in_dtype == LA_F32 || a->in_dtype == LA_BF16 || a->in_dtype == LA_F16,
             "la_gate_select: q/k dtype");
  return LA_OK;
}
}  // namespace la

extern "C" size_t la_gate_select_workspace(const la_gate_select_args *a) {
  if (gs_validate(a) != LA_OK) return 0;
  return (size_t)gs_layout(a).bytes;
}

extern "C" int la_gate_select(const la_gate_select_args *a, void *stream) {
  int rc = gs_validate(a);
  if (rc != LA_OK) return rc;
  const GsLayout L = gs_layout(a);
  if (!a->workspace || a->ws_bytes < L.bytes)
    return fail(LA_ERR_WORKSPACE, "la_gate_select: workspace %lld < %lld bytes",
                (long long)a->ws_bytes, (long long)L.bytes);
  hipStream_t st = (hipStream_t)stream;
  char *ws = (char *)a->workspace;
  double *kbar = (double *)(ws + L.kbar_off);
  double *sc = (double *)(ws + L.sc_off);
  if (a->kbar) {  // block means kept by the caller (la_block_means)
    kbar = const_cast<double *>(a->kbar);
  } else {
    pool_rows(a->k, a->in_dtype, a->B, a->Hkv, a->T, a->D, a->k_sb, a->k_sh, a->k_st, a->block,
              L.nkb, kbar, st);
    LA_LAUNCHED();
  }
  ScKP sp{};
  sp.q = a->q;
  sp.q_dt = a->in_dtype;
  sp.q_sb = a->q_sb;
  sp.q_sh = a->q_sh;
  sp.q_st = a->q_st;
  sp.kbar = kbar;
  sp.scores = sc;
  sp.Hq = a->Hq;
  sp.Hkv = a->Hkv;
  sp.nq = a->Tq;
  sp.nkb = L.nkb;
  sp.D = a->D;
  sp.pos0 = a->offset;
  sp.qunit = 1;
  sp.kunit = a->block;
  block_scores(sp, a->B, st);
  LA_LAUNCHED();
  TopkKParams tp{};
  tp.scores = sc;
  tp.row_stride = L.nkb;
  tp.G = 1;
  tp.Tq = a->Tq;
  tp.NG = a->B * a->Hq * a->Tq;
  tp.t_base = 0;
  tp.out_tq = a->Tq;
  tp.n = L.nkb;
  tp.k = a->topk;
  tp.width = a->width;
  tp.pos_off = a->offset;  // visible: block start <= offset + t; own = (offset + t) / block
  tp.pos_unit = a->block;
  tp.sink = 0;
  tp.window = 1;  // the own block, OR'd after the top-k (selection.py:632-633)
  tp.order = 1;
  tp.out_idx = a->out_idx;
  tp.out_count = a->out_count;
  return topk_launch(tp, st);
}

// ------------------------------------------------------------ block means --
namespace la {
static int bm_validate(const la_block_means_args *a) {
  LA_REQUIRE(a && a->k && a->out, "la_block_means: null pointer");
  LA_REQUIRE(a->B > 0 && a->H > 0 && a->T > 0 && a->D > 0 && a->block > 0,
             "la_block_means: bad shape");
  LA_REQUIRE(a->in_dtype == LA_F32 || a->in_dtype == LA_BF16 || a->in_dtype == LA_F16,
             "la_block_means: k dtype");
  const int64_t nkb = ceil_div(a->T, a->block);
  if (!a->positions)
    LA_REQUIRE(a->first_block >= 0 && a->n_blocks >= 0 && a->first_block + a->n_blocks <= nkb,
               "la_block_means: blocks [%lld, %lld) outside [0, %lld)", (long long)a->first_block,
               (long long)(a->first_block + a->n_blocks), (long long)nkb);
  LA_REQUIRE(nkb < ((int64_t)1 << 31) && a->B < 65536 && a->H < 65536, "la_block_means: grid");
  return LA_OK;
}
}  // namespace la

extern "C" int la_block_means(const la_block_means_args *a, void *stream) {
  const int rc = bm_validate(a);
  if (rc != LA_OK) return rc;
  const int64_t nkb = ceil_div(a->T, a->block);
  const int64_t npool = a->positions ? 1 : a->n_blocks;
  if (npool == 0) return LA_OK;
  pool_rows(a->k, a->in_dtype, a->B, a->H, a->T, a->D, a->k_sb, a->k_sh, a->k_st, a->block, nkb,
            a->out, (hipStream_t)stream, a->lengths, a->positions ? 0 : a->first_block, npool,
            a->positions);
  LA_LAUNCHED();
  return LA_OK;
}
