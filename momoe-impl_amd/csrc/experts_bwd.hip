// Backward of the experts, data-gradient side: dL/dh (before the gate weight), the SwiGLU
// backward for rows whose pre-activations were saved (the others get theirs in the epilogue of
// the recomputing x.Wl1 GEMM), dL/dx in sorted order, and the scatter of the gate-weight
// gradient into [N, M].
#include <algorithm>

#include "dgrad_h.hpp"
#include "dgrad_x.hpp"
#include "gemm_span.hpp"
#include "gs_tokens.hpp"

namespace momoe {
namespace {

// Both data-gradient GEMMs take WideSpan tiles (takes_span_tiles).  The rest go to the kernels of gemm_tile.hpp that
// hold narrow tiles, and wide ones where the table has too many for those (narrow_tiles_fit).

// u = G_y[idx] . Wl2^T: both operands are k-contiguous (k = D).
struct DhSpan {
  using G = WideSpan;
  static constexpr bool EXCHANGE = false;
  using Rows = SpanGatheredRows<256>;
  using Weights = SpanPitchedRows<G::COLS>;
  using Ids = FetchIds;
  struct Late {};
  const DhArgs& p;
  const int K, n_org;

  __device__ __forceinline__ explicit DhSpan(const DhArgs& p_)
      : p(p_), K(p_.D), n_org(wave_id() % G::WCOLS * (16 * G::FN)) {}
  __device__ __forceinline__ void gather(const TileCoord& t, Ids& g) const { g.gather(t, p.idx); }
  __device__ __forceinline__ void late(const TileCoord&, const Ids&, Late&) const {}
  __device__ __forceinline__ void settle(Ids& g) const { momoe::settle(g.tok); }
  __device__ __forceinline__ void settle(Late&) const {}
  __device__ __forceinline__ void setup(const TileCoord& t, const Ids& g, Rows& A, Weights& W) const {
    A.init(p.gy, [&](int j, int l) { return (uint32_t)g.of(j, l) * (uint32_t)(2 * p.D); });
    W.init(p.w2 + (int64_t)t.expert * p.H * p.D, p.D, t.tn * G::COLS, p.H);
  }
  template <int NA>
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x4 (&acc)[G::FN][NA], const Ids&, const Late&,
                                           bf16* staging) const {
    store_rows(acc, staging, p.u, (int64_t)tc.row0 + tc.mbase, tc.rows - tc.mbase, p.H, tc.tn * G::COLS + n_org,
               fresh_lane(), [](int) { return 1.0f; });
  }
};

__global__ __launch_bounds__(kSpanThreads, 1) void dgrad_h_kernel(DhArgs p) {
  const ClockTrace trace(p.clk);
  run_span_tiles<DhSpan>(p, (p.H + WideSpan::COLS - 1) / WideSpan::COLS, MOMOE_TILE_ROWS);
  trace.finish();
}

__device__ __forceinline__ void dgrad_h_by_table(const DhArgs& p) {
  if (TileSched::tile_rows_of(p.table) > StdTiles::MAX_ROWS) dgrad_h_tiles<TallTiles>(p);
  else dgrad_h_tiles<StdTiles>(p);
}
__global__ __launch_bounds__(kThreads, 2) void dgrad_h_narrow_kernel(DhArgs p) {
  const ClockTrace trace(p.clk);
  if (__builtin_expect(narrow_tiles_fit(p.table, (p.H + NarrowTiles::COLS - 1) / NarrowTiles::COLS), 1))
    dgrad_h_tiles<NarrowTiles, OneGeometrySched<NarrowTiles>>(p);
  else
    dgrad_h_by_table(p);
  trace.finish();
}
constexpr size_t kDhLds = std::max(DhProg<TallTiles>::Ring::BYTES, DhProg<StdTiles>::Ring::BYTES);
constexpr size_t kDhNarrowLds = std::max(DhProg<NarrowTiles>::Ring::BYTES, kDhLds);

// SwiGLU backward for the sorted rows whose a|b were saved by the forward.  One workgroup per
// group of 32 padded sorted rows (an expert's rows start at a multiple of 32 in padded
// positions, so a group never straddles two experts); it walks the hidden columns 64 at a time:
// thread t holds row t/8 and 8 of the 64 columns, writes its piece of gz row-major, and passes
// its piece of hs through LDS transposed, from where 8 consecutive rows of one column leave per
// thread for the transposed copy of hs.  Rows of the group past the expert's last one become the zero padding.
// A group belongs to this kernel when all of its rows lie below `Msave`; the remaining groups
// (those of the expert that Msave cuts, from the group holding Msave on, and all later experts)
// are produced by momoe_lin1_swiglu_bwd, which applies the same rule.
// Bound by HBM; a|b and u are read here for the last time.  ONCE (kBeyondCache): 65536 rows, H = 1024
// (778 MB in and out) 147 -> 134 us = 5.8 TB/s.
struct SavedArgs {
  const bf16* ab;
  const bf16* u;
  const float* s;
  int64_t ssn, ssm;
  const int32_t* idx;
  const int32_t* cumsums;
  bf16* gz;
  bf16* hst;
  int64_t ldt;
  float* gs_part;
  int nparts;
  int64_t msum, msave;
  int H, N, M;
};

constexpr int kSavedCols = 64;    // hidden columns per pass
constexpr int kSavedSpan = 256;   // hidden columns per workgroup: blockIdx.y selects the span
static_assert(kSavedSpan % MOMOE_GS_BLOCK == 0 && kSavedSpan % kSavedCols == 0, "spans cover whole parts");

template <bool ONCE>
__global__ __launch_bounds__(256) void swiglu_bwd_saved_kernel(SavedArgs p) {
  __shared__ __attribute__((aligned(16))) bf16 tr[2][kSavedCols * 32];  // [pass parity][column][row]
  const int H = p.H, N = p.N;
  const int pg = blockIdx.x * 32;  // first padded position of the group
  // expert whose padded range holds pg: the last e with padded_start(cumsums[e], e) <= pg
  int lo = 0, hi = N;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (padded_start(min(p.cumsums[mid], (int)p.msum), mid) <= pg) lo = mid; else hi = mid;
  }
  const int c0 = min(p.cumsums[lo], (int)p.msum), c1 = min(p.cumsums[lo + 1], (int)p.msum);
  const int local = pg - padded_start(c0, lo);  // rows of the expert before this group
  const int valid = min(32, c1 - c0 - local);   // rows of the group that exist
  if (local < 0 || valid <= 0) return;           // padding between two experts
  const int64_t r0 = (int64_t)c0 + local;        // first sorted row of the group
  if (r0 + valid > p.msave) return;              // not (entirely) below the save boundary

  const int t = threadIdx.x, row = t >> 3, cc = (t & 7) * 8;
  const bool rowok = row < valid;
  const int64_t r = r0 + min(row, valid - 1);
  const int tok = min(max(p.idx[r], 0), p.M - 1);
  const float sv = p.s[(int64_t)lo * p.ssn + (int64_t)tok * p.ssm];
  const bf16* a_row = p.ab + r * 2 * H;
  const bf16* u_row = p.u + r * H;
  float gsum = 0.0f;
  int par = 0;
  const int hbeg = blockIdx.y * kSavedSpan, hend = min(H, hbeg + kSavedSpan);
  for (int h0 = hbeg; h0 < hend; h0 += kSavedCols, par ^= 1) {
    const int c = h0 + cc;
    bf16x8 hv = {0, 0, 0, 0, 0, 0, 0, 0};
    if (c < H) {
      const bf16x8 a8 = load_maybe_once<ONCE>((const bf16x8*)(a_row + c));
      const bf16x8 b8 = load_maybe_once<ONCE>((const bf16x8*)(a_row + H + c));
      const bf16x8 u8 = load_maybe_once<ONCE>((const bf16x8*)(u_row + c));
      bf16x8 ga, gb;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float a = (float)a8[e], b = (float)b8[e], u = (float)u8[e];
        const float sg = sigmoidf_fast(b);
        const float hval = a * b * sg;
        gsum += u * hval;
        const float gh = sv * u;
        ga[e] = (bf16)(gh * b * sg);
        gb[e] = (bf16)(gh * a * sg * (1.0f + b * (1.0f - sg)));
        hv[e] = (bf16)(rowok ? sv * hval : 0.0f);
      }
      if (rowok) {  // gz is k-blocked: [2H/32][Msum][32]
        *(bf16x8*)(p.gz + ((int64_t)(c >> 5) * p.msum + r) * 32 + (c & 31)) = ga;
        *(bf16x8*)(p.gz + ((int64_t)((H + c) >> 5) * p.msum + r) * 32 + (c & 31)) = gb;
      }
    }
    // transposed staging: column-major, the four 8-row groups of a column rotated by the
    // column so that the 8 threads of a row (columns 8 apart) do not share a bank
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int col = cc + e;
      tr[par][col * 32 + (((row >> 3) ^ (col >> 3)) & 3) * 8 + (row & 7)] = hv[e];
    }
    __syncthreads();  // one barrier per pass: the other buffer is rewritten only after the next one
    const int col = t >> 2, rg = t & 3;
    if (h0 + col < H) {
      const bf16x8 v = *(const bf16x8*)(&tr[par][col * 32 + ((rg ^ (col >> 3)) & 3) * 8]);
      *(bf16x8*)(p.hst + ((int64_t)blockIdx.x * p.ldt + h0 + col) * 32 + rg * 8) = v;
    }
  }
  // dL/ds of the row: the 8 threads of a row are consecutive lanes
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) gsum += __shfl_xor(gsum, o);
  // the sum over this workgroup's span goes to part blockIdx.y; the parts that no span owns
  // (there are ceil(H/128) parts and ceil(H/256) spans) are zeroed by the first span
  if (rowok && (t & 7) == 0) p.gs_part[(int64_t)blockIdx.y * p.msum + r] = gsum;
  if (blockIdx.y == 0 && rowok)
    for (int q = gridDim.y + (t & 7); q < p.nparts; q += 8) p.gs_part[(int64_t)q * p.msum + r] = 0.0f;
}

// gxs = gz . Wl1^T: contraction over the 2H contiguous columns of both operands.
struct DxSpan {
  using G = WideSpan;
  static constexpr bool EXCHANGE = false;
  using Rows = SpanBlockedRows<256>;
  using Weights = SpanPitchedRows<G::COLS>;
  struct Ids {};
  struct Late {};
  const DxArgs& p;
  const int K, n_org;

  __device__ __forceinline__ explicit DxSpan(const DxArgs& p_)
      : p(p_), K(2 * p_.H), n_org(wave_id() % G::WCOLS * (16 * G::FN)) {}
  __device__ __forceinline__ void gather(const TileCoord&, Ids&) const {}
  __device__ __forceinline__ void late(const TileCoord&, const Ids&, Late&) const {}
  __device__ __forceinline__ void settle(Ids&) const {}
  __device__ __forceinline__ void settle(Late&) const {}
  __device__ __forceinline__ void setup(const TileCoord& t, const Ids&, Rows& A, Weights& W) const {
    A.init(p.gz, p.msum, t.row0, t.rows);
    W.init(p.w1 + (int64_t)t.expert * p.D * K, K, t.tn * G::COLS, p.D);
  }
  template <int NA>
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x4 (&acc)[G::FN][NA], const Ids&, const Late&,
                                           bf16* staging) const {
    store_rows(acc, staging, p.gxs, (int64_t)tc.row0 + tc.mbase, tc.rows - tc.mbase, p.D, tc.tn * G::COLS + n_org,
               fresh_lane(), [](int) { return 1.0f; });
  }
};

__global__ __launch_bounds__(kSpanThreads, 1) void dgrad_x_kernel(DxArgs p) {
  const ClockTrace trace(p.clk);
  run_span_tiles<DxSpan>(p, (p.D + WideSpan::COLS - 1) / WideSpan::COLS, MOMOE_TILE_ROWS);
  trace.finish();
}

__global__ __launch_bounds__(kThreads, 2) void dgrad_x_narrow_kernel(DxArgs p) { dgrad_x_short(p); }

// dL/ds [N][M] from the partial row sums in sorted order.  One workgroup per (expert, kGsTokens
// tokens) writes its piece whole, zeros included, through LDS: every line of the matrix is stored
// once (scattering into a matrix cleared beforehand took a launch more and stored the lines of the
// pairs twice: 9.8 + 8.2 us at 8192 tokens x 128 experts).  An expert's rows ascend in token, so
// one probe of its rows by all threads bounds those that belong to the piece.
constexpr int kGsTokens = 2048;

__global__ __launch_bounds__(256) void gs_scatter_kernel(const float* __restrict__ part, int nparts,
                                                         const int32_t* __restrict__ idx,
                                                         const int32_t* __restrict__ cumsums,
                                                         float* __restrict__ gs, int M, int N,
                                                         int64_t msum) {
  __shared__ float piece[kGsTokens];
  const int t = threadIdx.x, expert = blockIdx.y;
  const int m0 = blockIdx.x * kGsTokens, m1 = min(M, m0 + kGsTokens);
  // more pairs than rows: the routing was refused (empty tile table), dL/ds is zero
  const int limit = cumsums[N] > msum ? 0 : (int)msum;
  const int c0 = min(cumsums[expert], limit), rows = min(cumsums[expert + 1], limit) - c0;
  const int step = (rows + 255) / 256;
  const int probe = t * step;
  const int tok = rows > 0 ? idx[c0 + min(probe, rows - 1)] : 0;
  for (int m = t; m < kGsTokens; m += 256) piece[m] = 0.0f;
  // probes below the piece, and below its end: rows outside [lo, hi) hold tokens outside it
  const int below = __syncthreads_count(probe < rows && tok < m0);
  const int before_end = __syncthreads_count(probe < rows && tok < m1);
  const int lo = max(below - 1, 0) * step, hi = min(rows, before_end * step);
  for (int r = lo + t; r < hi; r += 256) {
    const int m = idx[c0 + r];
    if (m < m0 || m >= m1) continue;
    float v = 0.0f;
    for (int q = 0; q < nparts; ++q) v += part[(int64_t)q * msum + c0 + r];
    piece[m - m0] = v;
  }
  __syncthreads();
  for (int m = m0 + t; m < m1; m += 256) gs[(int64_t)expert * M + m] = piece[m - m0];
}

__global__ __launch_bounds__(kGsThreads) void gs_scatter_tokens_kernel(GsTokensArgs p) {
  __shared__ GsTile tile;
  gs_scatter_tokens(p, blockIdx.x, blockIdx.y, tile);
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

inline int check_dims(int64_t M, int64_t D, int64_t H, int64_t N, int64_t Msum) {
  if (M <= 0 || D <= 0 || H <= 0 || N <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  if (D % kBK != 0 || H % kBK != 0) return MOMOE_ERR_UNSUPPORTED;
  // per-lane source offsets are 32-bit byte offsets from G_y / from an expert's weights
  if (Msum >= (1ll << 31) || M * D * 2 >= (1ll << 32) || D * H * 4 >= (1ll << 32))
    return MOMOE_ERR_UNSUPPORTED;
  return MOMOE_OK;
}

}  // namespace
}  // namespace momoe

using namespace momoe;

extern "C" int momoe_dgrad_h(const void* Gy_MD, const void* Wl2_NHD, const int32_t* idx_Msum,
                             const int32_t* tile_table, void* u_MsumH, int64_t M, int64_t D,
                             int64_t H, int64_t N, int64_t Msum, void* stream) {
  if (!Gy_MD || !Wl2_NHD || !idx_Msum || !tile_table || !u_MsumH) return MOMOE_ERR_BAD_ARG;
  if (!aligned16(Gy_MD) || !aligned16(Wl2_NHD) || !aligned16(u_MsumH)) return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  DhArgs a{(const bf16*)Gy_MD, (const bf16*)Wl2_NHD, idx_Msum, tile_table, (bf16*)u_MsumH, (int)D,
           (int)H, clock_trace_buffer()};
  if (takes_span_tiles(Msum, N, H, D)) {
    static LdsLimit span;
    return launch_span(dgrad_h_kernel, a, span, (hipStream_t)stream);
  }
  static LdsLimit narrow;
  if (!allow_lds(dgrad_h_narrow_kernel, kDhNarrowLds, narrow)) return MOMOE_ERR_LAUNCH;
  dgrad_h_narrow_kernel<<<persistent_grid(), kThreads, kDhNarrowLds, (hipStream_t)stream>>>(a);
  return launch_status();
}

extern "C" int momoe_swiglu_bwd_saved(const void* ab_save, const void* u_MsumH, const float* s_NM,
                                      int64_t s_stride_n, int64_t s_stride_m,
                                      const int32_t* idx_Msum, const int32_t* cumsums_N1,
                                      int64_t Msave, void* gz_blocked, void* hsT_GH32,
                                      int64_t ld_hsT, float* gs_part, int64_t nparts, int64_t M,
                                      int64_t H, int64_t N, int64_t Msum, void* stream) {
  if (!ab_save || !u_MsumH || !s_NM || !idx_Msum || !cumsums_N1 || !gz_blocked || !hsT_GH32 ||
      !gs_part)
    return MOMOE_ERR_BAD_ARG;
  if (Msave < 0 || Msave > Msum || nparts <= 0 || M <= 0 || H <= 0 || N <= 0 || Msum <= 0)
    return MOMOE_ERR_BAD_ARG;
  if (!aligned16(ab_save) || !aligned16(u_MsumH) || !aligned16(gz_blocked) || !aligned16(hsT_GH32))
    return MOMOE_ERR_BAD_ARG;
  const int64_t mpad = momoe_padded_rows(Msum, N);
  if (ld_hsT < H || ld_hsT % 8 != 0) return MOMOE_ERR_BAD_ARG;
  if (H % 8 != 0 || mpad >= (1ll << 31) || M >= (1ll << 31) || nparts > (1 << 20))
    return MOMOE_ERR_UNSUPPORTED;
  if (Msave == 0) return MOMOE_OK;
  SavedArgs a{(const bf16*)ab_save, (const bf16*)u_MsumH, s_NM, s_stride_n, s_stride_m, idx_Msum,
              cumsums_N1, (bf16*)gz_blocked, (bf16*)hsT_GH32, ld_hsT, gs_part, (int)nparts, Msum,
              Msave, (int)H, (int)N, (int)M};
  const int64_t spans = cdiv64(H, kSavedSpan);
  if (spans > nparts || spans > 65535) return MOMOE_ERR_BAD_ARG;  // nparts = ceil(H / MOMOE_GS_BLOCK)
  auto kernel = Msave * 3 * H * 2 >= kBeyondCache ? swiglu_bwd_saved_kernel<true> : swiglu_bwd_saved_kernel<false>;
  kernel<<<dim3((unsigned)(mpad / 32), (unsigned)spans), 256, 0, (hipStream_t)stream>>>(a);
  return launch_status();
}

extern "C" int momoe_gs_scatter(const float* gs_part, int64_t nparts, const int32_t* idx_Msum,
                                const int32_t* cumsums_N1, float* Gs_NM, int64_t M, int64_t N,
                                int64_t Msum, void* stream) {
  if (!gs_part || !idx_Msum || !cumsums_N1 || !Gs_NM) return MOMOE_ERR_BAD_ARG;
  if (nparts <= 0 || M <= 0 || N <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  if (Msum >= (1ll << 31) || M >= (1ll << 31) - kGsTokens || N > 65535) return MOMOE_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)cdiv64(M, kGsTokens), (unsigned)N);
  gs_scatter_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(
      gs_part, (int)nparts, idx_Msum, cumsums_N1, Gs_NM, (int)M, (int)N, Msum);
  return launch_status();
}

extern "C" int momoe_gs_scatter_tokens(const float* gs_part, int64_t nparts, const int32_t* idx_Msum,
                                       const int32_t* cumsums_N1, float* Gs_MN, int64_t M, int64_t N,
                                       int64_t Msum, void* stream) {
  if (!gs_part || !idx_Msum || !cumsums_N1 || !Gs_MN) return MOMOE_ERR_BAD_ARG;
  if (nparts <= 0 || M <= 0 || N <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  const int64_t across = cdiv64(N, kGsTileExperts);
  if (Msum >= (1ll << 31) || M >= (1ll << 31) - kGsTileTokens || across > 65535) return MOMOE_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)cdiv64(M, kGsTileTokens), (unsigned)across);
  gs_scatter_tokens_kernel<<<grid, kGsThreads, 0, (hipStream_t)stream>>>(
      {gs_part, (int)nparts, idx_Msum, cumsums_N1, Gs_MN, (int)M, (int)N, Msum});
  return launch_status();
}

extern "C" int momoe_dgrad_x(const void* gz_blocked, const void* Wl1_ND2H,
                             const int32_t* tile_table, void* gxs_MsumD, int64_t M, int64_t D,
                             int64_t H, int64_t N, int64_t Msum, void* stream) {
  if (!gz_blocked || !Wl1_ND2H || !tile_table || !gxs_MsumD) return MOMOE_ERR_BAD_ARG;
  if (!aligned16(gz_blocked) || !aligned16(Wl1_ND2H) || ((uintptr_t)gxs_MsumD & 7))
    return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  DxArgs a{(const bf16*)gz_blocked, (const bf16*)Wl1_ND2H, tile_table, (bf16*)gxs_MsumD, (int)D,
           (int)H, Msum, clock_trace_buffer()};
  if (takes_span_tiles(Msum, N, D, 2 * H)) {
    static LdsLimit span;
    return launch_span(dgrad_x_kernel, a, span, (hipStream_t)stream);
  }
  static LdsLimit narrow;
  if (!allow_lds(dgrad_x_narrow_kernel, kDxNarrowLds, narrow)) return MOMOE_ERR_LAUNCH;
  dgrad_x_narrow_kernel<<<persistent_grid(), kThreads, kDxNarrowLds, (hipStream_t)stream>>>(a);
  return launch_status();
}
