// The gate-weight gradient in the layout of the gate weights: a launch of its own (experts_bwd.hip), and a part of the launch that
// ends the backward of a small call (wgrad.hip).
#pragma once
#include "common.hpp"

namespace momoe {
namespace {

// dL/ds [M][N] from the partial row sums in sorted order, the experts of a token next to each other, as a router that works on
// [tokens, experts] hands the gate weights over: a gradient in their layout needs no copy.  A workgroup writes a tile of
// 64 tokens x 16 experts whole, half a wavefront an expert.
// Bound by latency, a chain of prefix sum -> token of a row -> its partial sums: an expert of up to 256 rows is read
// as it is, a larger one probed at 32 places at a time until that many are left, and partial sums are loaded eight at
// a time.  In us, a scatter to [N][M] and the copy behind it -> this: 1024 tokens x 32 experts of 128 rows 9.1 -> 4.3, 8192 x 128
// of 512 18.5 -> 9.1, 16384 x 64, four of them with every token, 55 -> 10; 128 x 8 5.9 -> 2.8.
constexpr int kGsTileTokens = 64, kGsTileExperts = 16, kGsLanes = 32;
constexpr int kGsThreads = kGsLanes * kGsTileExperts;

struct GsTokensArgs {
  const float* part;  // [nparts][msum]
  int nparts;
  const int32_t *idx, *cumsums;
  float* gs;
  int M, N;
  int64_t msum;
};
typedef float GsTile[kGsTileTokens][kGsTileExperts + 1];

// tile (bx, by) of the result, through `tile` in LDS
__device__ __forceinline__ void gs_scatter_tokens(const GsTokensArgs& p, int bx, int by, GsTile& tile) {
  constexpr int THREADS = kGsThreads, ROUNDS = 8, AT_ONCE = 8;
  const int t = threadIdx.x, e = t / kGsLanes, s = t % kGsLanes, e0 = by * kGsTileExperts, expert = min(e0 + e, p.N - 1);
  const int m0 = bx * kGsTileTokens, m1 = min(p.M, m0 + kGsTileTokens);
  // more pairs than rows: the routing was refused (empty tile table), dL/ds is zero
  const int limit = p.cumsums[p.N] > p.msum ? 0 : (int)p.msum;
  const int c0 = min(p.cumsums[expert], limit), rows = e0 + e < p.N ? min(p.cumsums[expert + 1], limit) - c0 : 0;
  for (int i = t; i < kGsTileTokens * (kGsTileExperts + 1); i += THREADS) (&tile[0][0])[i] = 0.0f;
  int lo = 0, hi = rows;  // the rows of the tile's tokens, 64 at most, lie in [lo, hi)
  for (int probes = 0; probes < 6 && __any(hi - lo > ROUNDS * kGsLanes); ++probes) {
    const int step = (hi - lo + kGsLanes - 1) / kGsLanes, probe = lo + (s + 1) * step - 1;
    const bool is = step > 0 && probe < hi;
    const int m = is ? p.idx[c0 + probe] : m1;
    const int below = __popc((uint32_t)(__ballot(is && m < m0) >> (t & 32)));
    const int before_end = __popc((uint32_t)(__ballot(is && m < m1) >> (t & 32)));
    hi = min(hi, lo + (before_end + 1) * step);
    lo += below * step;
  }
  __syncthreads();
  for (; lo < hi; lo += ROUNDS * kGsLanes) {  // (once, if no token is listed twice)
    int m[ROUNDS];
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) m[j] = p.idx[c0 + min(lo + s + j * kGsLanes, hi - 1)];
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      const int r = lo + s + j * kGsLanes;
      if (r >= hi || m[j] < m0 || m[j] >= m1) continue;
      float v = 0.0f;
      for (int q0 = 0; q0 < p.nparts; q0 += AT_ONCE) {
        float v8[AT_ONCE];
#pragma unroll
        for (int q = 0; q < AT_ONCE; ++q) v8[q] = p.part[(int64_t)min(q0 + q, p.nparts - 1) * p.msum + c0 + r];
#pragma unroll
        for (int q = 0; q < AT_ONCE; ++q) v += q0 + q < p.nparts ? v8[q] : 0.0f;
      }
      tile[m[j] - m0][e] = v;
    }
  }
  __syncthreads();
  for (int i = t; i < kGsTileTokens * kGsTileExperts; i += THREADS) {
    const int m = m0 + i / kGsTileExperts, x = i % kGsTileExperts;
    if (m < p.M && e0 + x < p.N) p.gs[(int64_t)m * p.N + e0 + x] = tile[i / kGsTileExperts][x];
  }
}

}  // namespace
}  // namespace momoe
