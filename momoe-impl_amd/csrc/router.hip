// Top-k + softmax router with selection bias and shared experts: the elementwise
// part of the forward (everything after the gate GEMM) and the backward through
// renormalisation and softmax.  One wavefront per token (lane j holds columns
// j, j+64, ...), a workgroup per block of consecutive tokens so that the [N, M]
// tensors (mask, dL/ds) are touched in whole lines where that counts.  HBM-bound: a few
// passes over [M, N] fp32.
#include <type_traits>

#include "gate.hpp"

namespace momoe {
namespace {

constexpr int kMaxCols = 8;  // columns per lane -> N <= 512

// op over the wavefront, in every lane: lanes meet those 32, 16, 8, 4, 2 and 1 apart, by exchanges of the vector unit (through
// LDS a step is several times as long, and a token has four such chains).  Four apart: eight lanes apart hold the
// same by then, so the lane four further on in a row of 16 will do.  In us, through LDS -> this: forward 7.4 -> 7.1 (16
// tokens x 128 experts), backward 7.0 -> 5.8 (1000 x 128), 7.7 -> 6.4 (8192 x 128), 18.5 -> 15.5 (32768 x 96).
template <class Op>
__device__ __forceinline__ float wave_all(float v, Op op) {
  const auto swap = [&](auto pair) { return op(__uint_as_float(pair[0]), __uint_as_float(pair[1])); };
  v = swap(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  v = swap(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
  const auto lanes = [](auto ctrl, float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v = op(v, lanes(std::integral_constant<int, 0x128>{}, v));  // row_ror:8
  v = op(v, lanes(std::integral_constant<int, 0x124>{}, v));  // row_ror:4
  v = op(v, lanes(std::integral_constant<int, 0x4E>{}, v));   // quad_perm: lane ^ 2
  v = op(v, lanes(std::integral_constant<int, 0xB1>{}, v));   // quad_perm: lane ^ 1
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_all(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_all(v, [](float a, float b) { return a + b; });
}

// The maximum over the wavefront, in every lane, without LDS traffic: lanes exchange within quads
// and rows of 16, then a row's result passes to the rows above it; lane 63 ends up with all of it.
// fmaxf(v, v) where a lane has no source (bound_ctrl off keeps `old` = v).
template <int CTRL, int ROWS>
__device__ __forceinline__ float max_dpp(float v) {
  const int o = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xf, false);
  return fmaxf(v, __int_as_float(o));
}
__device__ __forceinline__ float wave_max_all(float v) {
  v = max_dpp<0xB1, 0xf>(v);   // quad_perm: lane ^ 1
  v = max_dpp<0x4E, 0xf>(v);   // quad_perm: lane ^ 2
  v = max_dpp<0x141, 0xf>(v);  // row_half_mirror: the other quad of 8 lanes
  v = max_dpp<0x140, 0xf>(v);  // row_mirror: the other half of 16 lanes
  v = max_dpp<0x142, 0xa>(v);  // row_bcast15: row 0 -> 1, row 2 -> 3
  v = max_dpp<0x143, 0xc>(v);  // row_bcast31: row 1 -> 2, 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Gate logits of few tokens: x . Wg split over the contraction, a workgroup for each 128 k-values of 128 experts and 64
// tokens; the router's kernel adds up the fp32 partial products and rounds the sums to bf16, as a product of its own would.
// Bound by the latency of one round of loads; with many tokens by the partial sums, so up to kGateMaxRows rows and kGateMaxSums
// of them (8 MiB), and up to kGateMaxTokens, where the host's time for a library product stops to show.  Product and router in
// a graph, us, a library product -> this: 1 token, D = 2048, N = 128 10.3 -> 8.2, 16 10.7 -> 8.8, 64 17.4 -> 9.9, 512
// 11.7 -> 12.0, 1000 20.5 -> 14.3; 1000, 1024, 128 15.6 -> 12.2; 2048, 1024, 128 15.9 -> 14.9; 2048, 512, 16 8.0 -> 8.5;
// 2048, 128, 128 10.7 -> 11.7; 512, 1024, 256 15.2 -> 15.0; 256, 1024, 512 19.3 -> 20.8.  Whole calls, H = 64, K = 4,
// forward | forward and backward, below the line: 2000, 512, 256 52.2 -> 50.8 | 201 -> 174; 512, 2048, 256 81.7 -> 79.8 | 283 -> 273; 256, 2048, 512 171.9 -> 167.8 |
// 511 -> 503; above it: 2000, 1024, 256 67.6 -> 72.3 | 220 -> 216; 1000, 2048, 256 85.1 -> 88.6 | 291 -> 285; 2000, 1024, 512
// 131.4 -> 143.1 | 380 -> 379.  Past the tokens and rows, in a graph: 2000, 2048, 64 14.6 -> 15.4; 4096, 2048, 128 23.9 -> 30.4.
constexpr int64_t kGateMaxTokens = 2048, kGateMaxRows = 16 * 1024, kGateMaxSums = kGateMaxRows * 128;
constexpr int kGateTokens = 64, kGateDepth = 2 * GateStage::ROWS;

struct GateFwdArgs {
  const bf16* x;
  int64_t ldx;
  const bf16* wg;
  float* part;  // [parts][M][N]
  int M, D, N;
};

__global__ __launch_bounds__(GateStage::THREADS) void gate_logits_kernel(GateFwdArgs p) {
  constexpr int FM = kGateTokens / 16, FN = 2;  // fragments of a wavefront: all tokens, 32 experts
  __shared__ __attribute__((aligned(16))) bf16 sw[2 * GateStage::ELEMS];
  const int k0 = blockIdx.x * kGateDepth, n0 = blockIdx.y * GateStage::COLS, m0 = blockIdx.z * kGateTokens;
  const int l = threadIdx.x & 63, n_org = 32 * wave_id();
  GateStage w[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) w[s].load(p.wg + n0, p.N, min(GateStage::COLS, p.N - n0), k0 + s * GateStage::ROWS, p.D);
  // k-values 8 * (lane / 16) .. +7 of a token are 16 consecutive bytes; those past the end meet zeros of Wg, so they
  // have to be finite: zeros, too
  bf16x8 xf[kGateDepth / 32][FM];
#pragma unroll
  for (int h = 0; h < kGateDepth / 32; ++h)
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int k = k0 + 32 * h + 8 * (l >> 4);
      const bf16x8 v = *(const bf16x8*)(p.x + (int64_t)min(m0 + 16 * i + (l & 15), p.M - 1) * p.ldx + min(k, p.D - 8));
      xf[h][i] = k < p.D ? v : bf16x8{};
    }
  w[0].put(sw);
  w[1].put(sw + GateStage::ELEMS);
  __syncthreads();
  if (n0 + n_org >= p.N) return;  // wave-uniform
  f32x4 acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int h = 0; h < kGateDepth / 32; ++h)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const bf16x8 wf = GateStage::frag(sw + (h / 2) * GateStage::ELEMS, n_org + 16 * j, h % 2);
#pragma unroll
      for (int i = 0; i < FM; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[h][i], acc[j][i], 0, 0, 0);
    }
  // a lane holds, for one token (lane % 16), experts 4 * (lane / 16) .. +3
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + 16 * i + (l & 15);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + n_org + 16 * j + 4 * (l >> 4);
      if (m < p.M && n < p.N) *(f32x4*)(p.part + ((int64_t)blockIdx.x * p.M + m) * p.N + n) = acc[j][i];
    }
  }
}

struct RouterFwdArgs {
  const void* logits;
  int logits_f32;
  int parts;  // PARTS: `logits` are that many fp32 partial sums [parts][M][N], the logits their sums in bf16
  const float* bias;
  int M, N, K, Ks;
  int32_t* mask;
  float* s;
  float* psel;
  float* ng;
  float* ks;
};

// A workgroup handles kTok consecutive tokens.  The mask is [N, M] (token fastest)
// while everything else is per token: the 0/1 flags of the tokens go through LDS and leave as
// rows of kTok x 4 bytes (written per token they would be N scattered 4-byte stores each).  With
// 32 tokens, two per wavefront, these are whole 128-byte lines; up to kRouterOneEach tokens, where
// 16-token workgroups still find a CU each, a wavefront takes one token and the second one's
// latency is saved.  Up to kRouterSpread tokens a workgroup is four wavefronts with a token each: the vector instructions of
// the rounds count then, and 16 tokens keep one CU busy where four could share them; the mask leaves in pieces of 16 bytes, an
// eighth of a line, which its size at that many tokens (1.5 MiB of 128 experts) allows.  In us, 16 tokens a workgroup -> 4:
// 16 tokens x 128 experts, K = 8 7.1 -> 5.1, 1000 x 128 7.6 -> 5.8, 2048 x 128 7.8 -> 6.6, 3000 x 64, K = 4 5.0 -> 4.7,
// 4096 x 64, K = 6 5.0 -> 5.5.
constexpr int kRouterThreads = 1024;
constexpr int64_t kRouterOneEach = 256 * 16, kRouterSpread = 3072;
static_assert(kGateMaxTokens <= kRouterSpread, "partial sums are taken by the workgroups of four tokens");

// NC = columns held per lane (1, 2, 4 or 8): N <= 64 * NC
// PARTS: the logits are partial sums.
template <int NC, int kTok, int THREADS = kRouterThreads, bool PARTS = false>
__global__ __launch_bounds__(THREADS) void router_fwd_kernel(RouterFwdArgs p) {
  __shared__ uint8_t flags[64 * NC][kTok];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int N = p.N, Ng = p.N - p.Ks, Kg = p.K - p.Ks;
  const int ncol = (N + 63) >> 6;
  const int m0 = blockIdx.x * kTok;
  for (int tt = wave; tt < kTok; tt += THREADS / 64) {
    const int m = m0 + tt;
    if (m >= p.M) break;  // wave-uniform
    float v[NC], pr[NC], score[NC], bias[NC];
    bool sel[NC];
    float mg = -INFINITY, ms = -INFINITY;
    // unconditional loads (column clamped, result masked): loads under a branch would be
    // waited for one by one
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int jc = min(lane + 64 * min(c, ncol - 1), N - 1);
      bias[c] = p.bias[jc];
      if constexpr (PARTS) {
        constexpr int AT_ONCE = 16;
        const float* part = (const float*)p.logits + (int64_t)m * N + jc;
        float sum = 0.0f;
        for (int q0 = 0; q0 < p.parts; q0 += AT_ONCE) {
          float t[AT_ONCE];
#pragma unroll
          for (int q = 0; q < AT_ONCE; ++q) t[q] = part[(int64_t)min(q0 + q, p.parts - 1) * p.M * N];
#pragma unroll
          for (int q = 0; q < AT_ONCE; ++q) sum += q0 + q < p.parts ? t[q] : 0.0f;
        }
        v[c] = (float)(bf16)sum;
      } else {
        v[c] = p.logits_f32 ? ((const float*)p.logits)[(int64_t)m * N + jc] : (float)((const bf16*)p.logits)[(int64_t)m * N + jc];
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      if (c < ncol && j < N) {
        if (j < Ng) mg = fmaxf(mg, v[c]); else ms = fmaxf(ms, v[c]);
      } else {
        v[c] = -INFINITY;
      }
    }
    mg = wave_max(mg);
    if (p.Ks > 0) ms = wave_max(ms);  // (uniform; nothing to exchange without shared experts)
    float sg = 0.0f, ss = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      pr[c] = 0.0f;
      if (c < ncol && j < N) {
        pr[c] = expf(v[c] - (j < Ng ? mg : ms));
        if (j < Ng) sg += pr[c]; else ss += pr[c];
      }
    }
    sg = wave_sum(sg);
    if (p.Ks > 0) ss = wave_sum(ss);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      sel[c] = false;
      score[c] = -INFINITY;
      if (c < ncol && j < N) {
        pr[c] = pr[c] / (j < Ng ? sg : ss);
        if (j < Ng) score[c] = pr[c] + bias[c];
      }
    }
    // top-Kg of score over the routed columns; ties go to the lower column.  A round is bound by
    // the latency of its cross-lane steps: the highest score left travels through the vector
    // unit's lane permutations (wave_max_all), and its lowest column comes from one ballot per 64
    // columns (carrying (score, column) pairs through LDS permutes took twelve dependent LDS round
    // trips a round).
    // Measured with 128 experts, K = 8: 16 tokens 10.9 -> 8.0 us, 1000 tokens 20.7 -> 9.2.
    for (int round = 0; round < Kg; ++round) {
      float best = -INFINITY;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (!sel[c]) best = fmaxf(best, score[c]);
      best = wave_max_all(best);
      bool found = false;  // wave-uniform
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const bool is = !sel[c] && lane + 64 * c < Ng && score[c] == best;
        const uint64_t who = __ballot(is);
        if (!found && who != 0 && lane == __ffsll((unsigned long long)who) - 1) sel[c] = true;
        found = found || who != 0;
      }
    }
    float ngsum = 0.0f, kssum = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      if (c < ncol && j < N) {
        if (j < Ng) ngsum += sel[c] ? pr[c] : 0.0f; else kssum += pr[c];
      }
    }
    ngsum = wave_sum(ngsum);
    if (p.Ks > 0) kssum = wave_sum(kssum);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      if (c < ncol && j < N) {
        const bool routed = j < Ng;
        const bool on = routed ? sel[c] : true;
        const float pv = on ? pr[c] : 0.0f;
        p.psel[(int64_t)m * N + j] = pv;
        p.s[(int64_t)m * N + j] = routed ? pv / ngsum : pv / kssum;
        flags[j][tt] = on ? 1 : 0;
      }
    }
    if (lane == 0) {
      p.ng[m] = ngsum;
      p.ks[m] = kssum;
    }
  }
  __syncthreads();
  // mask rows: kTok tokens x 4 bytes per expert
  const int tt = threadIdx.x & (kTok - 1);
  if (m0 + tt < p.M)
    for (int j = threadIdx.x / kTok; j < N; j += THREADS / kTok)
      p.mask[(int64_t)j * p.M + m0 + tt] = flags[j][tt];
}

struct RouterBwdArgs {
  const float* gs;
  int64_t gsn, gsm;
  const float* psel;
  const float* s;
  const float* ng;
  const float* ks;
  const int32_t* mask;
  int M, N, Ks;
  bf16* out;
};

// TB consecutive tokens per workgroup of 16 wavefronts.  dL/ds and the mask are [N, M]: a token's
// column is N scattered 4-byte reads, so the TB columns are first copied to LDS with loads that
// run along whichever index is contiguous in memory, and the per-token pass reads them there.
template <int TB, int NC>
__global__ __launch_bounds__(kRouterThreads) void router_bwd_kernel(RouterBwdArgs p) {
  constexpr int kTileFloats = 512 * 17;  // N <= 512 with TB = 16 (8704), N <= 256 with TB = 32 (8448)
  static_assert(TB == 32 || TB == 16, "tile sizes the LDS arrays are cut for");
  __shared__ float gs_t[kTileFloats];       // [N][TB + 1]
  __shared__ uint8_t mk_t[256 * 32];        // [N][TB]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int N = p.N, Ng = p.N - p.Ks;
  const int ncol = (N + 63) >> 6;
  const int m0 = blockIdx.x * TB;
  const int ntok = min(TB, p.M - m0);
  if (p.gsm == 1) {  // tokens contiguous: [N, M] as the experts' backward writes it
    for (int q = threadIdx.x; q < N * TB; q += kRouterThreads) {
      const int j = q / TB, tt = q % TB;
      if (tt < ntok) gs_t[j * (TB + 1) + tt] = p.gs[(int64_t)j * p.gsn + m0 + tt];
    }
  } else {           // any other strides: run along the experts
    for (int q = threadIdx.x; q < N * TB; q += kRouterThreads) {
      const int tt = q / N, j = q % N;
      if (tt < ntok) gs_t[j * (TB + 1) + tt] = p.gs[(int64_t)j * p.gsn + (int64_t)(m0 + tt) * p.gsm];
    }
  }
  for (int q = threadIdx.x; q < N * TB; q += kRouterThreads) {
    const int j = q / TB, tt = q % TB;
    if (tt < ntok) mk_t[j * TB + tt] = p.mask[(int64_t)j * p.M + m0 + tt] != 0;
  }
  __syncthreads();
  for (int tt = wave; tt < ntok; tt += kRouterThreads / 64) {
    const int m = m0 + tt;
    float g[NC], pv[NC], sv[NC];
    float dotg = 0.0f, dots = 0.0f;
    // unconditional loads (column clamped, results masked), all issued before any is used
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int jc = min(lane + 64 * min(c, ncol - 1), N - 1);
      pv[c] = p.psel[(int64_t)m * N + jc];
      sv[c] = p.s[(int64_t)m * N + jc];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      g[c] = 0.0f;
      if (c < ncol && j < N) {
        g[c] = gs_t[j * (TB + 1) + tt];
        if (j < Ng) dotg += mk_t[j * TB + tt] ? g[c] * sv[c] : 0.0f;
        else dots += g[c] * sv[c];
      } else {
        pv[c] = 0.0f;
      }
    }
    dotg = wave_sum(dotg);
    dots = wave_sum(dots);
    const float ing = 1.0f / p.ng[m];
    const float iks = p.Ks > 0 ? 1.0f / p.ks[m] : 0.0f;
    float o[NC];
    float inner_g = 0.0f, inner_s = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      o[c] = 0.0f;
      if (c < ncol && j < N) {
        if (j < Ng) {
          o[c] = (g[c] - dotg) * ing;
          inner_g += o[c] * pv[c];
        } else {
          o[c] = (g[c] - dots) * iks;
          inner_s += o[c] * pv[c];
        }
      }
    }
    inner_g = wave_sum(inner_g);
    inner_s = wave_sum(inner_s);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = lane + 64 * c;
      if (c < ncol && j < N)
        p.out[(int64_t)m * N + j] = (bf16)(pv[c] * (o[c] - (j < Ng ? inner_g : inner_s)));
    }
  }
}

// biases += rate * sign(c_avg - sizes): the auxiliary-loss-free balancing step
__global__ __launch_bounds__(256) void bias_update_kernel(const int64_t* __restrict__ sizes, float c_avg,
                                                          float rate, int N, float* __restrict__ biases) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  const float d = c_avg - (float)sizes[i];
  biases[i] += rate * (d > 0.0f ? 1.0f : d < 0.0f ? -1.0f : 0.0f);
}

}  // namespace
}  // namespace momoe

using namespace momoe;

static int launch_router_fwd(const RouterFwdArgs& a, hipStream_t st) {
  const int64_t M = a.M, N = a.N;
  auto by_width = [&](auto one, auto two, auto four, auto eight) { return N <= 64 ? one : N <= 128 ? two : N <= 256 ? four : eight; };
  if (M <= kRouterSpread) {
    auto kernel = a.parts > 0 ? by_width(router_fwd_kernel<1, 4, 256, true>, router_fwd_kernel<2, 4, 256, true>,
                                         router_fwd_kernel<4, 4, 256, true>, router_fwd_kernel<8, 4, 256, true>)
                              : by_width(router_fwd_kernel<1, 4, 256>, router_fwd_kernel<2, 4, 256>, router_fwd_kernel<4, 4, 256>,
                                         router_fwd_kernel<8, 4, 256>);
    kernel<<<(unsigned)cdiv64(M, 4), 256, 0, st>>>(a);
    return launch_status();
  }
  const bool few = M <= kRouterOneEach;
  auto kernel = few ? by_width(router_fwd_kernel<1, 16>, router_fwd_kernel<2, 16>, router_fwd_kernel<4, 16>, router_fwd_kernel<8, 16>)
                    : by_width(router_fwd_kernel<1, 32>, router_fwd_kernel<2, 32>, router_fwd_kernel<4, 32>, router_fwd_kernel<8, 32>);
  kernel<<<(unsigned)cdiv64(M, few ? 16 : 32), kRouterThreads, 0, st>>>(a);
  return launch_status();
}

static int check_router_fwd(int64_t M, int64_t N, int64_t K, int64_t Ks) {
  if (M <= 0 || N <= 0 || Ks < 0 || K < Ks || Ks > N || K - Ks > N - Ks) return MOMOE_ERR_BAD_ARG;
  return N > 64 * kMaxCols || M >= (1ll << 31) - 4 ? MOMOE_ERR_UNSUPPORTED : MOMOE_OK;
}

extern "C" int momoe_router_fwd(const void* logits_MN, int logits_f32, const float* biases_N,
                                int64_t M, int64_t N, int64_t K, int64_t Ks, int32_t* mask_NM,
                                float* s_MN, float* p_sel_MN, float* Ng_M, float* Ks_M,
                                void* stream) {
  if (!logits_MN || !biases_N || !mask_NM || !s_MN || !p_sel_MN || !Ng_M || !Ks_M)
    return MOMOE_ERR_BAD_ARG;
  const int status = check_router_fwd(M, N, K, Ks);
  if (status != MOMOE_OK) return status;
  return launch_router_fwd({logits_MN, logits_f32, 0, biases_N, (int)M, (int)N, (int)K, (int)Ks, mask_NM, s_MN, p_sel_MN, Ng_M, Ks_M},
                           (hipStream_t)stream);
}

extern "C" int64_t momoe_gate_router_workspace_bytes(int64_t M, int64_t D, int64_t N) {
  if (M <= 0 || D <= 0 || N <= 0 || D % 8 != 0 || N % 8 != 0 || N > 64 * kMaxCols || D > (1 << 20) || M > kGateMaxTokens ||
      cdiv64(D, kGateDepth) * M > kGateMaxRows || cdiv64(D, kGateDepth) * M * N > kGateMaxSums)
    return -1;
  return cdiv64(D, kGateDepth) * M * N * (int64_t)sizeof(float);
}

extern "C" int momoe_gate_router_fwd(const void* x_MD, int64_t ldx, const void* Wg_DN, const float* biases_N, int64_t M, int64_t D,
                                     int64_t N, int64_t K, int64_t Ks, int32_t* mask_NM, float* s_MN, float* p_sel_MN, float* Ng_M,
                                     float* Ks_M, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x_MD || !Wg_DN || !biases_N || !mask_NM || !s_MN || !p_sel_MN || !Ng_M || !Ks_M || !workspace) return MOMOE_ERR_BAD_ARG;
  const int status = check_router_fwd(M, N, K, Ks);
  if (status != MOMOE_OK) return status;
  if (D <= 0 || ldx < D) return MOMOE_ERR_BAD_ARG;
  const int64_t need = momoe_gate_router_workspace_bytes(M, D, N);
  if (need < 0 || ldx % 8 != 0) return MOMOE_ERR_UNSUPPORTED;
  if (workspace_bytes < need || ((uintptr_t)x_MD & 15) || ((uintptr_t)Wg_DN & 15) || ((uintptr_t)workspace & 15))
    return MOMOE_ERR_BAD_ARG;
  hipStream_t st = (hipStream_t)stream;
  const GateFwdArgs g{(const bf16*)x_MD, ldx, (const bf16*)Wg_DN, (float*)workspace, (int)M, (int)D, (int)N};
  const dim3 grid((unsigned)cdiv64(D, kGateDepth), (unsigned)cdiv64(N, GateStage::COLS), (unsigned)cdiv64(M, kGateTokens));
  gate_logits_kernel<<<grid, GateStage::THREADS, 0, st>>>(g);
  const int launched = launch_status();
  if (launched != MOMOE_OK) return launched;
  return launch_router_fwd({workspace, 1, (int)grid.x, biases_N, (int)M, (int)N, (int)K, (int)Ks, mask_NM, s_MN, p_sel_MN, Ng_M, Ks_M},
                           st);
}

extern "C" int momoe_router_bwd(const float* Gs_NM, int64_t gs_stride_n, int64_t gs_stride_m,
                                const float* p_sel_MN, const float* s_MN, const float* Ng_M,
                                const float* Ks_M, const int32_t* mask_NM, int64_t M, int64_t N,
                                int64_t Ks, void* Glogits_MN, void* stream) {
  if (!Gs_NM || !p_sel_MN || !s_MN || !Ng_M || !Ks_M || !mask_NM || !Glogits_MN)
    return MOMOE_ERR_BAD_ARG;
  if (M <= 0 || N <= 0 || Ks < 0 || Ks > N) return MOMOE_ERR_BAD_ARG;
  if (N > 64 * kMaxCols || M >= (1ll << 31) - 4) return MOMOE_ERR_UNSUPPORTED;
  RouterBwdArgs a{Gs_NM, gs_stride_n, gs_stride_m, p_sel_MN, s_MN, Ng_M, Ks_M, mask_NM,
                  (int)M, (int)N, (int)Ks, (bf16*)Glogits_MN};
  hipStream_t st = (hipStream_t)stream;
  const unsigned grid32 = (unsigned)cdiv64(M, 32);
  if (N <= 64) router_bwd_kernel<32, 1><<<grid32, kRouterThreads, 0, st>>>(a);
  else if (N <= 128) router_bwd_kernel<32, 2><<<grid32, kRouterThreads, 0, st>>>(a);
  else if (N <= 256) router_bwd_kernel<32, 4><<<grid32, kRouterThreads, 0, st>>>(a);
  else router_bwd_kernel<16, 8><<<(unsigned)cdiv64(M, 16), kRouterThreads, 0, st>>>(a);
  return launch_status();
}

extern "C" int momoe_bias_update(const int64_t* sizes_N, float c_avg, float rate, int64_t N,
                                 float* biases_N, void* stream) {
  if (!sizes_N || !biases_N || N <= 0) return MOMOE_ERR_BAD_ARG;
  if (N >= (1ll << 31) - 256) return MOMOE_ERR_UNSUPPORTED;
  bias_update_kernel<<<(unsigned)cdiv64(N, 256), 256, 0, (hipStream_t)stream>>>(sizes_N, c_avg, rate, (int)N, biases_N);
  return launch_status();
}
