// Totals of what lists read, for the variants' read accounting.
#include <algorithm>

#include "common.h"

namespace la {

struct LrKP {
  const int32_t *ids, *counts;
  int64_t id_sb, id_sh, id_st, L, Tq, W, rep, unit, offset, t_k, rows, n_counts;
  uint64_t *totals;
  int32_t lw;  // log2 of the lanes of a row
};

// 2^lw lanes per row (at least its entries, at most a wave); the same totals as
// torch's masks and sums over the expanded lists, which took ten launches and two
// host reads per call: 150 us of a 256-query chunk, about 5 us and no host read
// here.  Every workgroup writes a pair of its own, and the first one zeros the
// pairs past the grid: sums in one pair took a launch of 3.7 us that cleared it.
__global__ __launch_bounds__(256) void list_reads_kernel(LrKP p) {
  __shared__ uint64_t part[2][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lw = p.lw, per = 256 >> lw;  // rows of a workgroup at a time
  uint64_t reads = 0, cnt = 0;
  constexpr int NR = 8;  // rows of a thread read before they are counted
  const int64_t step = (int64_t)gridDim.x * per;
  const int e0 = threadIdx.x & ((1 << lw) - 1);
  for (int64_t r0 = (int64_t)blockIdx.x * per + (threadIdx.x >> lw); r0 < p.rows; r0 += NR * step) {
    const int32_t *list[NR];
    int64_t lim[NR];
    int32_t id[NR];
#pragma unroll
    for (int x = 0; x < NR; ++x) {
      const int64_t r = min(r0 + x * step, p.rows - 1);
      const uint32_t q = (uint32_t)r / (uint32_t)p.Tq, t = (uint32_t)r - q * (uint32_t)p.Tq;
      const uint32_t b = q / (uint32_t)p.L, h = q - b * (uint32_t)p.L;
      list[x] = p.ids + b * p.id_sb + h * p.id_sh + (t / (uint32_t)p.rep) * p.id_st;
      lim[x] = r0 + x * step < p.rows ? min(p.offset + (int64_t)t + 1, p.t_k) : 0;
      id[x] = e0 < p.W ? list[x][e0] : -1;
    }
    for (int64_t e = e0; e < p.W; e += 1 << lw) {
#pragma unroll
      for (int x = 0; x < NR; ++x)
        if (id[x] >= 0) reads += (uint64_t)min(max(lim[x] - id[x] * p.unit, (int64_t)0), p.unit);
      const int64_t en = e + (1 << lw);
#pragma unroll
      for (int x = 0; x < NR; ++x) id[x] = en < p.W ? list[x][en] : -1;
    }
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < p.n_counts; i += (int64_t)gridDim.x * 256)
    cnt += (uint64_t)(int64_t)p.counts[i];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    reads += __shfl_xor(reads, o, 64);
    cnt += __shfl_xor(cnt, o, 64);
  }
  if (lane == 0) {
    part[0][w] = reads;
    part[1][w] = cnt;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const uint64_t s = part[threadIdx.x][0] + part[threadIdx.x][1] + part[threadIdx.x][2] + part[threadIdx.x][3];
    p.totals[2 * blockIdx.x + threadIdx.x] = s;
  }
  if (blockIdx.x == 0)
    for (int i = 2 * gridDim.x + threadIdx.x; i < 2 * LA_LIST_READS_PARTS; i += 256) p.totals[i] = 0;
}

}  // namespace la

using namespace la;

extern "C" int la_list_reads(const int32_t *ids, int64_t id_sb, int64_t id_sh, int64_t id_st, int64_t B,
                             int64_t L, int64_t Tq, int64_t W, int64_t rep, int64_t unit, int64_t offset,
                             int64_t t_k, const int32_t *counts, int64_t n_counts, uint64_t *totals,
                             void *stream) {
  LA_REQUIRE(ids && totals, "la_list_reads: null pointer");
  LA_REQUIRE(B > 0 && L > 0 && Tq > 0 && W > 0 && rep > 0 && unit > 0 && t_k >= 0, "la_list_reads: bad shape");
  const int64_t rows = B * L * Tq;
  LA_REQUIRE(rows < ((int64_t)1 << 31) && rep < ((int64_t)1 << 31), "la_list_reads: 2^31 rows or more");
  LA_REQUIRE(n_counts >= 0 && (counts || n_counts == 0), "la_list_reads: counts");
  LrKP p{ids, counts, id_sb, id_sh, id_st, L, Tq, W, rep, unit, offset, t_k, rows, n_counts, totals, 0};
  p.lw = std::min(6, ilog2(W));
  // As many workgroups as give a thread its rows at a time.
  const int64_t turns = ceil_div(rows, 256 >> p.lw) * ceil_div(W, (int64_t)1 << p.lw);
  const unsigned grid = (unsigned)std::min<int64_t>(LA_LIST_READS_PARTS, ceil_div(turns, 8));
  list_reads_kernel<<<dim3(grid), 256, 0, (hipStream_t)stream>>>(p);
  LA_LAUNCHED();
  return LA_OK;
}
