// Gradients of the router's gate product.
//
// Of the weights: G_Wg [D,N] = x^T . G_logits, a contraction over the tokens with few columns.
//
// Bound by memory: x is read once for every 128 experts, and that is nearly all there is.  The product has few tiles and a
// long contraction, so the tokens are split: a workgroup takes 128 columns of x, 128 experts and a range of tokens, and a
// second launch adds up the fp32 partial products of the ranges.  As many ranges as give every CU a workgroup, and no more than one
// for every 256 tokens begun.  Both launches in a graph, us, with half as many ranges | as they are | twice as many, and the library's product:
// 8192 tokens, D = 2048, N = 128 25.9 | 20.5 | 25.1, 59.3; 16384, 2048, 64 36.8 | 25.0 | 25.4, 89.9; 32768, 512, 16 22.2 | 18.7 |
// 21.6, 72.4; 7680, 2176, 64 23.5 | 17.1 | 19.8, 44.8.
// One range (of up to 256 tokens, or of any number in more than 128 tiles) is all of the product: no partial sums, which leaves the
// workspace as it is, and no second launch, which a call of few tokens, bound by the host, waits for.  Steps with their
// router, us, two launches -> one: 64 tokens, D = 256, N = 16 178.0 -> 171.9; 200, 1024, 32 186.0 -> 179.6.
#include <algorithm>

#include "gate.hpp"

namespace momoe {
namespace {

constexpr int kGateThreads = GateStage::THREADS, kTile = GateStage::COLS, kStageRows = GateStage::ROWS;
// 4 wavefronts, 2 x 2, each 64 x 64 of the tile in 4 x 4 accumulators

struct GateArgs {
  const bf16* x;
  int64_t ldx;
  const bf16* g;
  float* part;  // [ranges][D][N]
  bf16* out;    // [D][N] where one range is all: it is stored rounded, and nothing is left to add up
  int M, D, N, rows;  // rows: tokens of a range, a multiple of kStageRows
};

__global__ __launch_bounds__(kGateThreads, 2) void gate_wgrad_kernel(GateArgs p) {
  __shared__ __attribute__((aligned(16))) bf16 sx[GateStage::ELEMS], sg[GateStage::ELEMS];
  const int d0 = blockIdx.x * kTile, n0 = blockIdx.y * kTile;
  const int begin = blockIdx.z * p.rows, end = min(p.M, begin + p.rows);
  const int w = wave_id(), d_org = 64 * (w >> 1), n_org = 64 * (w & 1), l = threadIdx.x & 63;
  const bool some = n0 + n_org < p.N && d0 + d_org < p.D;  // wave-uniform
  const bf16 *x = p.x + d0, *g = p.g + n0;
  const int xcols = min(kTile, p.D - d0), gcols = min(kTile, p.N - n0);
  f32x4 acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // two stages are on their way while one is multiplied
  GateStage px[2], pg[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    px[s].load(x, p.ldx, xcols, begin + s * kStageRows, end);
    pg[s].load(g, p.N, gcols, begin + s * kStageRows, end);
  }
  for (int row = begin; row < end; row += 2 * kStageRows)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = row + s * kStageRows;
      if (at >= end) break;  // uniform
      px[s].put(sx);
      pg[s].put(sg);
      px[s].load(x, p.ldx, xcols, at + 2 * kStageRows, end);
      pg[s].load(g, p.N, gcols, at + 2 * kStageRows, end);
      __syncthreads();
      if (some) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          bf16x8 xf[4], gf[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) xf[i] = GateStage::frag(sx, d_org + 16 * i, h), gf[i] = GateStage::frag(sg, n_org + 16 * i, h);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gf[j], xf[i], acc[j][i], 0, 0, 0);
        }
      }
      __syncthreads();
    }
  if (!some) return;
  // a lane holds, for one column of x (lane % 16), experts 4 * (lane / 16) .. +3
  float* const out = p.part + (int64_t)blockIdx.z * p.D * p.N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = d0 + d_org + 16 * i + (l & 15);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + n_org + 16 * j + 4 * (l >> 4);
      if (d >= p.D || n >= p.N) continue;
      const f32x4 v = acc[j][i];
      if (p.out) store_bf16x4(p.out + (int64_t)d * p.N + n, v[0] + 0.0f, v[1] + 0.0f, v[2] + 0.0f, v[3] + 0.0f);
      else *(f32x4*)(out + (int64_t)d * p.N + n) = v;
    }
  }
}

// out = sum of the ranges' products, four elements a thread
__global__ __launch_bounds__(kGateThreads) void gate_wgrad_reduce_kernel(const float* __restrict__ part, int ranges, int64_t quads,
                                                                        bf16* __restrict__ out) {
  constexpr int AT_ONCE = 8;
  const int64_t q = (int64_t)blockIdx.x * kGateThreads + threadIdx.x;
  if (q >= quads) return;
  const f32x4* const p = (const f32x4*)part + q;
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int r0 = 0; r0 < ranges; r0 += AT_ONCE) {
    f32x4 v[AT_ONCE];
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r) v[r] = p[min(r0 + r, ranges - 1) * quads];
#pragma unroll
    for (int r = 0; r < AT_ONCE; ++r)
      if (r0 + r < ranges) sum += v[r];
  }
  ((bf16x4*)out)[q] = bf16x4{(bf16)sum[0], (bf16)sum[1], (bf16)sum[2], (bf16)sum[3]};
}

// Of the tokens: out [M,D] = G_x + G_logits . Wg^T, a contraction over the experts.  G_x in and the sum out are nearly all that
// has to move (8192 tokens, D = 2048, N = 128: 70 MB in 26 us, 2.7 TB/s, half of what a copy reaches): a wave waits for its
// fragments every 32 experts, and for its part of G_x behind them.  Both operands are k-contiguous and small
// enough for the caches, so fragments are loaded as they are, 64 x 64 a wavefront.
// A fragment's 16 rows of Wg are those of two runs of columns in turn, so that a lane holds 8 consecutive columns of a token and
// four lanes store 64 bytes.  In a graph, us, the library's product with its copy of G_x -> this: 128 tokens, D = 128, N = 8 10.3 ->
// 4.9; 1024, 1024, 32 7.3 -> 4.7; 2000, 1120, 48 14.5 -> 5.0; 8192, 2048, 128 32.7 -> 25.1; 32768, 512, 16 33.7 -> 13.8; 8192, 4096, 96
// 50.1 -> 31.8.
struct GateDgradArgs {
  const bf16 *gl, *wg, *gx;  // gx: nullptr if there is nothing to add
  bf16* out;
  int M, D, N;
};

__global__ __launch_bounds__(kGateThreads, 2) void gate_dgrad_kernel(GateDgradArgs p) {
  const int l = threadIdx.x & 63, r = l & 15, g = l >> 4, w = wave_id();
  const int d0 = blockIdx.x * kTile + 64 * (w & 1), m0 = blockIdx.y * kTile + 64 * (w >> 1);
  if (d0 >= p.D || m0 >= p.M) return;  // wave-uniform
  // fragment j: column r of it is column 32 (j / 2) + 8 (r / 4) + 4 (j % 2) + r % 4 of the wave's 64
  const bf16 *grow[4], *wrow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    grow[i] = p.gl + (int64_t)min(m0 + 16 * i + r, p.M - 1) * p.N;
    wrow[i] = p.wg + (int64_t)min(d0 + 32 * (i >> 1) + 8 * (r >> 2) + 4 * (i & 1) + (r & 3), p.D - 1) * p.N;
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int n0 = 0; n0 < p.N; n0 += 32) {
    const int n = n0 + 8 * g, at = min(n, p.N - 8);
    bf16x8 gf[4], wf[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) gf[i] = *(const bf16x8*)(grow[i] + at), wf[i] = *(const bf16x8*)(wrow[i] + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) gf[i] = n < p.N ? gf[i] : bf16x8{}, wf[i] = n < p.N ? wf[i] : bf16x8{};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], gf[i], acc[j][i], 0, 0, 0);
  }
  // a lane holds, for token r of fragment i, columns 32 q + 8 g .. +7 in fragments 2 q and 2 q + 1
  bf16x8 add[4][2];
  if (p.gx != nullptr) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        add[i][q] = *(const bf16x8*)(p.gx + (int64_t)min(m0 + 16 * i + r, p.M - 1) * p.D + min(d0 + 32 * q + 8 * g, p.D - 8));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (bf16)(acc[2 * q + e / 4][i][e % 4] + (p.gx != nullptr ? (float)add[i][q][e] : 0.0f));
      const int m = m0 + 16 * i + r, d = d0 + 32 * q + 8 * g;
      if (m < p.M && d < p.D) *(bf16x8*)(p.out + (int64_t)m * p.D + d) = o;
    }
}

struct GateSplit {
  int64_t rows, ranges;
  GateSplit(int64_t M, int64_t D, int64_t N) {
    const int64_t tiles = cdiv64(D, kTile) * cdiv64(N, kTile);
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>(256 / tiles, cdiv64(M, 4 * kStageRows)));
    rows = cdiv64(cdiv64(M, want), kStageRows) * kStageRows;
    ranges = cdiv64(M, rows);
  }
};

bool gate_sizes_ok(int64_t M, int64_t D, int64_t N) {
  return D % 8 == 0 && N % 8 == 0 && D <= (1 << 20) && N <= 4096 && M < (1ll << 31) - 4 * kStageRows && D * N < (1ll << 31);
}

}  // namespace
}  // namespace momoe

using namespace momoe;

extern "C" int64_t momoe_gate_wgrad_workspace_bytes(int64_t M, int64_t D, int64_t N) {
  if (M <= 0 || D <= 0 || N <= 0 || !gate_sizes_ok(M, D, N)) return -1;
  return GateSplit(M, D, N).ranges * D * N * (int64_t)sizeof(float);
}

extern "C" int momoe_gate_wgrad(const void* x_MD, int64_t ldx, const void* Glogits_MN, void* GWg_DN, int64_t M, int64_t D,
                                int64_t N, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x_MD || !Glogits_MN || !GWg_DN || !workspace) return MOMOE_ERR_BAD_ARG;
  if (M <= 0 || D <= 0 || N <= 0 || ldx < D) return MOMOE_ERR_BAD_ARG;
  if (!gate_sizes_ok(M, D, N) || ldx % 8 != 0) return MOMOE_ERR_UNSUPPORTED;
  if (((uintptr_t)x_MD & 15) || ((uintptr_t)Glogits_MN & 15) || ((uintptr_t)GWg_DN & 7) || ((uintptr_t)workspace & 15))
    return MOMOE_ERR_BAD_ARG;
  const GateSplit split(M, D, N);
  if (workspace_bytes < split.ranges * D * N * (int64_t)sizeof(float)) return MOMOE_ERR_BAD_ARG;
  hipStream_t st = (hipStream_t)stream;
  const GateArgs a{(const bf16*)x_MD, ldx, (const bf16*)Glogits_MN, (float*)workspace,
                   split.ranges == 1 ? (bf16*)GWg_DN : nullptr, (int)M, (int)D, (int)N, (int)split.rows};
  const dim3 grid((unsigned)cdiv64(D, kTile), (unsigned)cdiv64(N, kTile), (unsigned)split.ranges);
  gate_wgrad_kernel<<<grid, kGateThreads, 0, st>>>(a);
  const int status = launch_status();
  if (status != MOMOE_OK || split.ranges == 1) return status;
  const int64_t quads = D * N / 4;
  gate_wgrad_reduce_kernel<<<(unsigned)cdiv64(quads, kGateThreads), kGateThreads, 0, st>>>((const float*)workspace, (int)split.ranges,
                                                                                         quads, (bf16*)GWg_DN);
  return launch_status();
}

extern "C" int momoe_gate_dgrad(const void* Glogits_MN, const void* Wg_DN, const void* Gx_MD, void* out_MD, int64_t M, int64_t D,
                                int64_t N, void* stream) {
  if (!Glogits_MN || !Wg_DN || !out_MD || M <= 0 || D <= 0 || N <= 0) return MOMOE_ERR_BAD_ARG;
  if (!gate_sizes_ok(M, D, N) || cdiv64(M, kTile) > 65535) return MOMOE_ERR_UNSUPPORTED;
  for (const void* p : {Glogits_MN, Wg_DN, Gx_MD, (const void*)out_MD})
    if ((uintptr_t)p & 15) return MOMOE_ERR_BAD_ARG;
  const GateDgradArgs a{(const bf16*)Glogits_MN, (const bf16*)Wg_DN, (const bf16*)Gx_MD, (bf16*)out_MD, (int)M, (int)D, (int)N};
  const dim3 grid((unsigned)cdiv64(D, kTile), (unsigned)cdiv64(M, kTile));
  gate_dgrad_kernel<<<grid, kGateThreads, 0, (hipStream_t)stream>>>(a);
  return launch_status();
}
