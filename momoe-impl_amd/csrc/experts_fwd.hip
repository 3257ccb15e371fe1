// Forward of the experts: grouped GEMM x.Wl1 with fused SwiGLU, grouped GEMM
// h.Wl2 with the gate weight fused into the epilogue, and the K-way combine.
#include <algorithm>
#include <type_traits>

#include "dgrad_h.hpp"
#include "gemm_span.hpp"

namespace momoe {
namespace {

constexpr int FN = 2;  // 2x4 (4x2) waves, each (32 * FM) rows x 64 columns

struct Lin1Args {
  const bf16* x;
  const bf16* w1;
  const int32_t* idx;
  const int32_t* table;
  bf16* h;
  bf16* ab;
  int64_t ab_lo, ab_hi;
  int D, H;
  // backward only (rows >= ab_lo): dL/dh without the gate weight, the gate weights, outputs
  const bf16* u;
  const float* s;
  int64_t ssn, ssm;
  bf16* gz;
  bf16* hst;    // hs in groups of 32 padded sorted rows, [group][ldt features][32]
  int64_t ldt;
  float* gs_part;
  int64_t msum;
  unsigned long long* clk;
  // where u is made on the way (Lin1DhProg): G_y and Wl2
  const bf16* gy = nullptr;
  const bf16* w2 = nullptr;
};

// The forward.  Tile = up to 256 rows x (128 `a` columns + the matching 128 `b` columns); a wave's
// first half of fragments are `a` columns, the second their `b` columns, so the SwiGLU product pairs
// registers of the same lane.
struct Lin1Span {
  using G = WideSpan;
  static constexpr bool EXCHANGE = false;
  static constexpr int BNH = G::COLS / 2, WIDTH = 8 * G::FN;  // hidden columns of a tile, of a wave
  using Rows = SpanGatheredRows<256>;
  using Weights = SpanCols<true>;
  using Ids = FetchIds;
  struct Late {};
  const Lin1Args& p;
  const int K, n_org;

  __device__ __forceinline__ explicit Lin1Span(const Lin1Args& p_)
      : p(p_), K(p_.D), n_org(wave_id() % G::WCOLS * WIDTH) {}
  __device__ __forceinline__ void gather(const TileCoord& t, Ids& g) const { g.gather(t, p.idx); }
  __device__ __forceinline__ void late(const TileCoord&, const Ids&, Late&) const {}
  __device__ __forceinline__ void settle(Ids& g) const { momoe::settle(g.tok); }
  __device__ __forceinline__ void settle(Late&) const {}
  __device__ __forceinline__ void setup(const TileCoord& t, const Ids& g, Rows& A, Weights& W) const {
    const int D = p.D, H = p.H, j0 = t.tn * BNH;
    A.init(p.x, [&](int j, int l) { return (uint32_t)g.of(j, l) * (uint32_t)(2 * D); });
    W.init(p.w1 + (int64_t)t.expert * D * 2 * H, 2 * H,
           [&](int c) { return (c / BNH) * H + min(j0 + (c % BNH), H - 8); });
  }
  template <int NA>
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x4 (&acc)[G::FN][NA], const Ids&, const Late&,
                                           bf16* staging) const {
    constexpr int HF = G::FN / 2;
    using Stager = SpanStager<WIDTH>;
    const int H = p.H, j0 = tc.tn * BNH + n_org;  // first hidden column of this wave
    const Stager stager(staging, fresh_lane());
    const int rows = tc.rows - tc.mbase;
    const int64_t r0 = (int64_t)tc.row0 + tc.mbase;
    if (p.h) {
      keep_in_place(acc);
      // h is k-blocked for the next GEMM: 32 hidden columns of consecutive rows are one piece of memory
      bf16* const first = p.h + ((int64_t)(j0 >> 5) * p.msum + r0) * 32;  // uniform
      const uint32_t off = (stager.block_row() * 32 + stager.block_col()) * 2;
      bf16x8 v[2][Stager::PASSES];
      auto store = [&](int i) {
#pragma unroll
        for (int q = 0; q < Stager::PASSES; ++q)
          store16(first + ((int64_t)q * p.msum + 16 * i) * 32, off, 16 * i + stager.block_row() < rows && j0 + 32 * q < H,
                  v[i & 1][q]);
      };
#pragma unroll
      for (int i = 0; i < NA; ++i) {
#pragma unroll
        for (int f = 0; f < HF; ++f) {
          float hv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = acc[f][i][e], b = acc[HF + f][i][e];
            hv[e] = a * b * sigmoidf_fast(b);
          }
          stager.put(i & 1, f, pack_bf16x4(hv[0], hv[1], hv[2], hv[3]));
        }
        if (i > 0) store(i - 1);
#pragma unroll
        for (int q = 0; q < Stager::PASSES; ++q) v[i & 1][q] = stager.get_block(i & 1, q);
      }
      store(NA - 1);
    }
    if (p.ab) {
      keep_in_place(acc);
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
          for (int f = 0; f < HF; ++f) stager.put(half, f, pack_bf16x4(acc[half * HF + f][i], 1.0f));
#pragma unroll
          for (int q = 0; q < Stager::PASSES; ++q) {
            const int row = 16 * i + stager.row(q), col = j0 + stager.col(q);
            const bf16x8 v = stager.get(half, q);
            store16(p.ab + (r0 + 16 * i) * 2 * H + half * H + j0,
                    ((uint32_t)stager.row(q) * 2 * H + stager.col(q)) * 2,
                    row < rows && col < H && r0 + row >= p.ab_lo && r0 + row < p.ab_hi, v);
          }
        }
    }
  }
};

__global__ __launch_bounds__(kSpanThreads, 1) void lin1_swiglu_fwd_kernel(Lin1Args p) {
  const ClockTrace trace(p.clk);
  // without an h output only rows >= ab_lo are wanted: experts entirely below are skipped
  const int first = p.h == nullptr && p.ab_lo > 0 ? TileSched::expert_tile_of_row(p.table, p.ab_lo) : 0;
  using Prog = Lin1Span;
  run_span_tiles<Prog>(p, (p.H + Prog::BNH - 1) / Prog::BNH, MOMOE_TILE_ROWS, first);
  trace.finish();
}

// The recomputing backward (momoe/momoe.py:421-535), on the tiles of the forward: the a|b of the tile stay in registers and go
// straight into the SwiGLU backward.  With u = dL/dh before the gate weight s,  G_a = s u b sig(b),
// G_b = s u a sig(b) (1 + b (1 - sig(b))),  hs = s a b sig(b),  and the row sums of u a b sig(b) over the
// tile's 128 hidden columns.
struct Lin1BwdSpan {
  using G = WideSpan;
  static constexpr bool EXCHANGE = true;
  static constexpr int BNH = G::COLS / 2, WIDTH = 8 * G::FN, HF = G::FN / 2;
  static_assert(BNH == MOMOE_GS_BLOCK && G::WCOLS == 2, "a tile's row sums are one part, from two waves");
  using Rows = SpanGatheredRows<256>;
  using Weights = SpanCols<true>;
  using Stager = SpanStager<WIDTH>;
  struct Ids {
    FetchIds fetch;
    RowIds rows;  // of the accumulators
  };
  using Late = RowScales;
  const Lin1Args& p;
  const int K, n_org;

  __device__ __forceinline__ explicit Lin1BwdSpan(const Lin1Args& p_)
      : p(p_), K(p_.D), n_org(wave_id() % G::WCOLS * WIDTH) {}
  __device__ __forceinline__ void gather(const TileCoord& t, Ids& g) const { g.fetch.gather(t, p.idx), g.rows.gather(t, p.idx); }
  __device__ __forceinline__ void late(const TileCoord& t, const Ids& g, Late& l) const { l.load(t, g.rows, p.s, p.ssn, p.ssm); }
  __device__ __forceinline__ void settle(Ids& g) const { momoe::settle(g.fetch.tok), g.rows.settle(); }
  __device__ __forceinline__ void settle(Late& l) const { l.settle(); }
  __device__ __forceinline__ void setup(const TileCoord& t, const Ids& g, Rows& A, Weights& W) const {
    const int D = p.D, H = p.H, j0 = t.tn * BNH;
    A.init(p.x, [&](int j, int l) { return (uint32_t)g.fetch.of(j, l) * (uint32_t)(2 * D); });
    W.init(p.w1 + (int64_t)t.expert * D * 2 * H, 2 * H,
           [&](int c) { return (c / BNH) * H + min(j0 + (c % BNH), H - 8); });
  }
  // Rows below the save boundary are not this kernel's: the boundary is moved down to a multiple of 32
  // rows from the expert's first row (tiles start at such multiples), so that a whole group of 32 rows is
  // either produced here or by momoe_swiglu_bwd_saved.
  __device__ __forceinline__ int first_row(const TileCoord& tc) const {
    return p.ab_lo > tc.row0 ? (int)((p.ab_lo - tc.row0) & ~(int64_t)31) : 0;
  }
  // Staging areas: 0 G_a, 1 G_b, 2 and 3 hs of 32 rows.
  template <int NA>
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x4 (&acc)[G::FN][NA], const Ids&, const Late& scales,
                                           bf16* staging) const {
    static_assert(4 * Stager::ELEMS <= kStagingElems && NA % 2 == 0, "four areas; groups of 32 rows");
    const int H = p.H, j0 = tc.tn * BNH + n_org;  // first hidden column of this wave
    const int l = fresh_lane();
    const Stager stager(staging, l);
    const int rows = tc.rows - tc.mbase, lo = first_row(tc) - tc.mbase;
    const int64_t r0 = (int64_t)tc.row0 + tc.mbase;
    const bf16* const u0 = p.u + r0 * H;  // uniform
    bf16x4 uq[2][HF];
    auto load_u = [&](int i) {
      const uint32_t at = ((uint32_t)min(16 * i + (l & 15), rows - 1) * (uint32_t)H + 4 * (l >> 4)) * 2;
#pragma unroll
      for (int f = 0; f < HF; ++f) uq[i & 1][f] = *(const bf16x4*)((const char*)(u0 + (j0 + 16 * f < H ? j0 + 16 * f : 0)) + at);
    };
    // gz is k-blocked ([2H/32][Msum][32], the layout dL/dx contracts over): 32 columns of consecutive rows are one
    // piece of memory
    bf16* const gza = p.gz + ((int64_t)(j0 >> 5) * p.msum + r0) * 32;  // uniform
    const int64_t to_b = (int64_t)(H >> 5) * p.msum * 32;
    const uint32_t off = (stager.block_row() * 32 + stager.block_col()) * 2;
    bf16x8 v[2][2][Stager::PASSES];
    auto store_gz = [&](int i) {
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int q = 0; q < Stager::PASSES; ++q)
          store16(gza + half * to_b + ((int64_t)q * p.msum + 16 * i) * 32, off,
                  16 * i + stager.block_row() < rows && 16 * i >= lo && j0 + 32 * q < H, v[i & 1][half][q]);
    };
    // hs^T leaves as 8 consecutive rows of a column per lane.  Rows past the expert's last one are zeros: the
    // padding that the weight-gradient GEMM reads.
    bf16* const hst = p.hst + ((int64_t)((tc.prow0 + tc.mbase) >> 5) * p.ldt + j0) * 32;  // uniform
    const uint32_t hoff = (l & 15) * 64 + (l >> 4) * 16;
    bf16x8 hv[HF];
    auto store_hs = [&](int i) {
#pragma unroll
      for (int q = 0; q < HF; ++q)
        store16(hst + ((int64_t)(i / 2) * p.ldt + 16 * q) * 32, hoff, 16 * i >= lo && j0 + 16 * q < H, hv[q]);
    };
    load_u(0);
    float gsums[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      if (i + 1 < NA) load_u(i + 1);
      const float sv = scales.of(i, l);
      const bool some = 16 * i + (l & 15) < rows;
      float gsum = 0.0f;
#pragma unroll
      for (int f = 0; f < HF; ++f) {
        float va[4], vb[4], hs[4], part = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[f][i][e], b = acc[HF + f][i][e];
          const float u = (float)uq[i & 1][f][e];
          const float sg = sigmoidf_fast(b);
          const float t = b * sg;  // silu(b)
          const float hval = a * t;
          part += u * hval;
          const float gh = sv * u;
          va[e] = gh * t;
          // d silu / d b = sg (1 + b (1 - sg)) = sg + t - t sg
          vb[e] = (gh * a) * __builtin_fmaf(-t, sg, sg + t);
          hs[e] = some ? sv * hval : 0.0f;
        }
        if (j0 + 16 * f < H) gsum += part;
        momoe::settle(gsum);  // (summed up later, u and its factors were kept until then)
        stager.put(0, f, pack_bf16x4(va[0], va[1], va[2], va[3]));
        stager.put(1, f, pack_bf16x4(vb[0], vb[1], vb[2], vb[3]));
        stager.put(2 + (i & 1), f, pack_bf16x4(hs[0], hs[1], hs[2], hs[3]));
      }
      gsums[i] = gsum;
      if (i > 0) store_gz(i - 1);
      if (i > 0 && i % 2 == 0) store_hs(i - 1);
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int q = 0; q < Stager::PASSES; ++q) v[i & 1][half][q] = stager.get_block(half, q);
      if (i % 2 == 1) {
#pragma unroll
        for (int q = 0; q < HF; ++q) hv[q] = stager.get_rows(2, q);
      }
      order_fence();  // (loads of several rounds ahead were spilled)
    }
    store_gz(NA - 1);
    store_hs(NA - 1);
    // this wave's row sums, for finish()
    float* const red = (float*)(staging + wave_id() * kStagingElems);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      float g = gsums[i] + __shfl_xor(gsums[i], 16);
      g += __shfl_xor(g, 32);
      red[16 * i + (l & 15)] = g;  // (the same from four lanes)
    }
  }
  __device__ __forceinline__ void finish(const TileCoord& tc, bf16* staging) const {
    if (n_org != 0) return;  // wave-uniform: the other column half's wave is the next one
    const int l = fresh_lane(), lo = first_row(tc) - tc.mbase, rows = min(tc.rows - tc.mbase, 32 * tc.na);
    const float* const red = (const float*)(staging + wave_id() * kStagingElems);
    float* const part = p.gs_part + (int64_t)tc.tn * p.msum + tc.row0 + tc.mbase;  // uniform
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row = 64 * q + l;
      store4(part, row * 4, row < rows && row >= lo, red[row] + red[row + kStagingElems / 2]);
    }
  }
};

// Bound by the loop of gemm_span.hpp; the epilogue is some 6 us of a tile, of which the stores of gz (128 KB) and
// hs^T (64 KB) need 5 at the HBM's rate.
__global__ __launch_bounds__(kSpanThreads, 1) void lin1_swiglu_bwd_kernel(Lin1Args p) {
  const ClockTrace trace(p.clk);
  const int first = p.ab_lo > 0 ? TileSched::expert_tile_of_row(p.table, p.ab_lo) : 0;
  run_span_tiles<Lin1BwdSpan>(p, (p.H + Lin1BwdSpan::BNH - 1) / Lin1BwdSpan::BNH, WideSpan::MAX_ROWS, first);
  trace.finish();
}

// Whether a launch takes it rather than the 8 waves of Lin1Prog<true, StdTiles>: with as much work per workgroup
// as pays for the longer start and the last epilogue, about 3 us.  A tile costs 0.4 for its weights and 0.6 for
// 256 rows.
// Measured, there -> here in us: 65536 tokens, D = 4096, H = 2048, N = 64, K = 8 17297 -> 14150; 8192, 2048, 1024, 128, 8
// 664 -> 561; 7680, 2176, 1152, 64, 6 509 -> 437; 4000, 1024, 512, 64, 4 69 -> 57; 2048, 2048, 1024, 128, 8 (128
// rows per expert) 275 -> 267; in one round of tiles 3000, 3072, 1024, 32, 2 112 -> 102; 16000, 1024, 256, 128, 1
// (125 rows per expert, one round) 34 -> 38; 12000, 256, 128, 32, 4 21.6 -> 23.7.  At the line, D = 1024, H = 512: N = 64,
// 176 and 200 rows per expert 43 -> 49 and 44 -> 48; N = 32, 320, 400 and 512 rows 35 -> 34, 39 -> 40 and 71 -> 54.
// At most half a round, whose tiles are cut into pieces (SpanSched), pays off sooner: D = 1152, H = 64, N = 8, 269 rows 27 -> 20.
inline bool takes_span_recompute(int64_t msum, int64_t n, int64_t h, int64_t d) {
  if (d < WideSpan::AHEAD * kSpan || few_rows_per_expert(msum, n)) return false;
  const double mean = (double)msum / n, tiles = std::ceil(mean / WideSpan::MAX_ROWS);
  const double rounds = n * tiles * (double)cdiv64(h, Lin1BwdSpan::BNH) / persistent_grid();
  return std::max(1.0, rounds) * d * (0.4 + 0.6 * mean / (tiles * WideSpan::MAX_ROWS)) >= (rounds > 0.5 ? 900 : 780);
}

// Tile = up to 320 (256) rows x (128 `a` columns + the matching 128 `b` columns), or 64 + 64; a wave owns 32 `a`
// columns and their 32 `b` columns, so the SwiGLU product pairs registers of the same lane.
// BWD = false: forward / recomputation, writes h and/or a|b.  BWD = true: the a|b of the tile
// stay in registers and go straight into the SwiGLU backward.
// G: the row-tile geometry.  The forward takes either; the backward's epilogue needs the registers
// of the fifth fragment row, so it only exists for 256-row tiles and runs on a tile table of its own.
template <bool BWD, class G>
struct Lin1Prog {
  static_assert(!BWD || G::MAX_ROWS == StdTiles::MAX_ROWS, "the SwiGLU backward epilogue fits 256-row tiles only");
  static constexpr int FM = G::FM, BM = G::MAX_ROWS, BN = G::COLS;
  static constexpr bool MAY_ONCE = G::MAY_ONCE;
  using RowsOp = RDma<G::AROWS>;  // token rows, k-contiguous
  using WeightOp = TDmaT<BN, MAY_ONCE>;  // expert weights [k][col], k-strided
  using Ring = StageRing<RowsOp, WeightOp, G::STAGES>;
  static constexpr size_t kLds = Ring::BYTES;
  static constexpr int BNH = BN / 2;
  static_assert(!BWD || BNH == MOMOE_GS_BLOCK || 2 * BNH == MOMOE_GS_BLOCK, "gs_part blocks follow the hidden-column tile");
  static_assert(G::WCOLS * BM * sizeof(float) <= kEpilogueLds, "the dL/ds row sums reuse the staging area");
  struct Prep {
    int32_t tok[RowsOp::NCH];  // tokens of the rows this lane fetches
    int32_t etok[BWD ? FM : 1];  // backward: tokens of the rows this lane holds in the accumulators
    float sv[BWD ? FM : 1];      // and their gate weights
  };
  const Lin1Args& p;
  const int ktiles, wn;

  __device__ __forceinline__ void gather(const TileCoord& t, Prep& g) const {
#pragma unroll
    for (int j = 0; j < RowsOp::NCH; ++j) g.tok[j] = p.idx[t.row0 + min(RowsOp::row_of(j), t.rows - 1)];
    if (BWD) {
#pragma unroll
      for (int i = 0; i < FM; ++i) g.etok[i] = p.idx[t.row0 + min(t.mbase + 32 * i + acc_row(), t.rows - 1)];
    }
  }
  __device__ __forceinline__ void late(const TileCoord& t, Prep& g) const {
    if (BWD) {
#pragma unroll
      for (int i = 0; i < FM; ++i) g.sv[i] = p.s[(int64_t)t.expert * p.ssn + (int64_t)g.etok[i] * p.ssm];
    }
  }
  __device__ __forceinline__ void setup(const TileCoord& t, const Prep& g, RowsOp& A, WeightOp& B) const {
    const int D = p.D, H = p.H;
    const bf16* w = p.w1 + (int64_t)t.expert * D * 2 * H;
    const int j0 = t.tn * BNH;
    A.init(p.x, [&](int, int j) { return (uint32_t)g.tok[j] * (uint32_t)(2 * D); });
    B.init(w, [&](int c) { return (c / BNH) * H + min(j0 + (c % BNH), H - 8); }, 2 * H);
    if (MAY_ONCE) B.once = t.alone;
  }
  // epi: store staging; in the backward also the row-sum exchange
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x16 (&acc)[FN][FM], const Prep& g, bf16* epi) const {
    if (BWD) {
      const int H = p.H, j0 = tc.tn * BNH + wn * 32;
      epilogue_bwd(tc, acc, g, epi, [&](int i, bf16x4 (&uq)[4]) {
        const int64_t r = (int64_t)tc.row0 + min((tc.mbase + 32 * i) + acc_row(), tc.rows - 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) uq[q] = *(const bf16x4*)(p.u + r * H + min(j0 + acc_col(q), H - 4));
      });
    } else {
      epilogue_fwd(tc, acc, epi);
    }
  }

  __device__ __forceinline__ void epilogue_fwd(const TileCoord& tc, f32x16 (&acc)[FN][FM], bf16* epi) const {
    const int H = p.H;
    RowStager<1> stager(epi);
    const int j0 = tc.tn * BNH + wn * 32;  // first hidden column of this wave
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i >= tc.na) break;  // wave-uniform: no valid row in this fragment row
      float a[4][4], b[4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[q][e] = acc[0][i][4 * q + e];
          b[q][e] = acc[1][i][4 * q + e];
        }
      // destination of 8 columns of tile row (tc.mbase + 32 * i)+row in a [*, ld] matrix, or nullptr
      auto dst = [&](bf16* mat, int64_t ld, int col0, bool rows_lo_hi) {
        return [=, *this](int row, int col) -> bf16* {
          const int rl = (tc.mbase + 32 * i) + row;
          const int64_t r = (int64_t)tc.row0 + rl;
          if (rl >= tc.rows || j0 + col >= H) return nullptr;
          if (rows_lo_hi && (r < p.ab_lo || r >= p.ab_hi)) return nullptr;
          return mat + r * ld + col0 + j0 + col;
        };
      };
      if (p.h) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          stager.put(0, q, pack_bf16x4(a[q][0] * b[q][0] * sigmoidf_fast(b[q][0]),
                                       a[q][1] * b[q][1] * sigmoidf_fast(b[q][1]),
                                       a[q][2] * b[q][2] * sigmoidf_fast(b[q][2]),
                                       a[q][3] * b[q][3] * sigmoidf_fast(b[q][3])));
        // h is k-blocked for the next GEMM: this wave's 32 hidden columns are one k-block, so
        // the fragment's rows are consecutive 64-byte pieces of memory
        bf16* hblock = p.h + (int64_t)(j0 >> 5) * p.msum * 32;
        stager.flush([&](int row, int col) -> bf16* {
          const int rl = (tc.mbase + 32 * i) + row;
          if (rl >= tc.rows || j0 >= H) return nullptr;
          return hblock + ((int64_t)tc.row0 + rl) * 32 + col;
        });
      }
      if (p.ab) {
#pragma unroll
        for (int q = 0; q < 4; ++q) stager.put(0, q, pack_bf16x4(a[q][0], a[q][1], a[q][2], a[q][3]));
        stager.flush(dst(p.ab, 2 * H, 0, true));
#pragma unroll
        for (int q = 0; q < 4; ++q) stager.put(0, q, pack_bf16x4(b[q][0], b[q][1], b[q][2], b[q][3]));
        stager.flush(dst(p.ab, 2 * H, H, true));
      }
    }
  }

  // SwiGLU backward on the recomputed a|b (momoe/momoe.py:421-535): with u = dL/dh before the
  // gate weight s,  G_a = s u b sig(b),  G_b = s u a sig(b) (1 + b (1 - sig(b))),
  // hs = s a b sig(b),  and the partial row sum of u a b sig(b) over this tile's columns.  load_u(i, uq): the lane's u in
  // fragment row i.
  template <int NF, class LoadU>
  __device__ __forceinline__ void epilogue_bwd(const TileCoord& tc, f32x16 (&acc)[NF][FM], const Prep& g, bf16* epi, LoadU load_u) const {
    const int H = p.H;
    RowStager<1> stager(epi);
    float* red = (float*)epi;  // [column waves][BM]
    const int j0 = tc.tn * BNH + wn * 32;  // first hidden column of this wave
    RowStager<1> stager1(epi, 1);
    // Rows below the save boundary are not this kernel's: the boundary is moved down to a
    // multiple of 32 rows from the expert's first row (tiles start at such multiples), so that
    // a whole 32-row fragment row is either produced here or by momoe_swiglu_bwd_saved.
    const int rl_lo = p.ab_lo > tc.row0 ? (int)((p.ab_lo - tc.row0) & ~(int64_t)31) : 0;
    float gsums[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      gsums[i] = 0.0f;
      if (i >= tc.na) continue;  // wave-uniform
      bf16x4 uq[4];
      load_u(i, uq);
      const float sv = g.sv[i];
      float gsum = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float va[4], vb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[0][i][4 * q + e], b = acc[1][i][4 * q + e];
          const float u = (float)uq[q][e];
          const float sg = sigmoidf_fast(b);
          const float t = b * sg;  // silu(b)
          const float hval = a * t;
          gsum += u * hval;
          const float gh = sv * u;
          va[e] = gh * t;
          // d silu / d b = sg (1 + b (1 - sg)) = sg + t - t sg
          vb[e] = (gh * a) * __builtin_fmaf(-t, sg, sg + t);
          acc[0][i][4 * q + e] = sv * hval;  // a is not needed any more: keep hs in its place
        }
        stager.put(0, q, pack_bf16x4(va[0], va[1], va[2], va[3]));
        stager1.put(0, q, pack_bf16x4(vb[0], vb[1], vb[2], vb[3]));
      }
      const int rl0 = tc.mbase + 32 * i;  // first tile row of this fragment row
      const bool mine = rl0 >= rl_lo;      // wave-uniform
      // gz is k-blocked ([2H/32][Msum][32], the layout dL/dx contracts over): this wave's 32
      // columns of G_a are block j0/32, those of G_b block (H + j0)/32, and a fragment's rows are
      // consecutive 64-byte pieces of memory
      auto dst = [&](int block) {
        bf16* base = p.gz + (int64_t)block * p.msum * 32;
        return [=, *this](int row, int col) -> bf16* {
          const int rl = rl0 + row;
          if (rl >= tc.rows || j0 >= H || !mine) return nullptr;
          return base + ((int64_t)tc.row0 + rl) * 32 + col;
        };
      };
      stager.flush(dst(j0 >> 5));
      stager1.flush(dst((H + j0) >> 5));
      // hs^T: the 32 x 32 fragment goes through the staging area transposed ([column][row],
      // the four 8-row groups of a column permuted so that the two half-waves, which write
      // columns 4 apart, use different banks) and leaves it as 8 consecutive rows of one column
      // per lane.  Rows past the expert's last one are written as zeros: they are the padding
      // the weight-gradient GEMM reads.
      {
        bf16* tst = stager.st;
        const int row = acc_row();
        const bool rowok = rl0 + row < tc.rows;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int col = acc_col(q) + e;
            const int grp = (row >> 3) ^ ((col >> 2) & 3);
            tst[col * 32 + grp * 8 + (row & 7)] = (bf16)(rowok ? acc[0][i][4 * q + e] : 0.0f);
          }
        const int l = threadIdx.x & 63;
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
          const int col = pass * 16 + (l >> 2), rg = l & 3;
          const bf16x8 v = *(const bf16x8*)(tst + col * 32 + ((rg ^ ((col >> 2) & 3)) * 8));
          // the fragment's 32 columns x 32 rows are 2 KiB of consecutive memory
          if (mine && j0 + col < H)
            *(bf16x8*)(p.hst + ((int64_t)((tc.prow0 + rl0) >> 5) * p.ldt + j0 + col) * 32 + rg * 8) = v;
        }
      }
      // the wave's 32 hidden columns lie inside H or outside as a whole (H is a multiple of 32)
      gsums[i] = rl0 + acc_row() < tc.rows && j0 < H ? gsum : 0.0f;
    }
    // every wave is done with its staging area before the row sums overwrite it
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const float gg = gsums[i] + __shfl_xor(gsums[i], 32);
      // only the fragment rows this wave owns: the others belong to the other wave row
      if (i < tc.na && (threadIdx.x & 63) < 32) red[wn * BM + (tc.mbase + 32 * i) + acc_row()] = gg;
    }
    wait_lgkm0();  // the row sums are in LDS (a full fence would also wait for the stores above)
    __builtin_amdgcn_s_barrier();
    if ((int)threadIdx.x < tc.rows && (int)threadIdx.x >= rl_lo) {
      float sum = red[threadIdx.x];
#pragma unroll
      for (int w = 1; w < G::WCOLS; ++w) sum += red[w * BM + threadIdx.x];
      float* part = p.gs_part + (int64_t)tc.tn * (G::HALF_PARTS ? 2 : 1) * p.msum + tc.row0 + threadIdx.x;
      *part = sum;
      // (the columns' second half has its share in the first part)
      if (G::HALF_PARTS && j0 - wn * 32 + BNH / 2 < H) part[p.msum] = 0.0f;
    }
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();  // `red` is rewritten by the next tile
  }
};

template <bool BWD, class G, class Sched = TileSched>
__device__ __forceinline__ void lin1_swiglu_tiles(const Lin1Args& p) {
  using Prog = Lin1Prog<BWD, G>;
  using Ring = typename Prog::Ring;
  constexpr int FM = Prog::FM;
  Ring ring(dyn_lds());
  // without an h output only rows >= ab_lo are wanted: experts entirely below are skipped
  const int first_tile =
      p.h == nullptr && p.ab_lo > 0 ? Sched::expert_tile_of_row(p.table, p.ab_lo) : 0;
  Sched sched(p.table, (p.H + Prog::BNH - 1) / Prog::BNH, BWD ? Prog::BM : MOMOE_TILE_ROWS, first_tile);
  const int wn = wave_id() % G::WCOLS;
  const int n_org[FN] = {wn * 32, Prog::BNH + wn * 32};
  Prog prog{p, p.D / kBK, wn};
  run_row_tiles<FM, FN>(prog, sched, ring, n_org);
}

// The wide tiles: Short for tables of at most 256 rows, the forward also the tall ones.
template <bool BWD, class Short>
__device__ __forceinline__ void lin1_swiglu_by_table(const Lin1Args& p) {
  if constexpr (BWD) {
    lin1_swiglu_tiles<true, Short>(p);
  } else {
    if (TileSched::tile_rows_of(p.table) > Short::MAX_ROWS) lin1_swiglu_tiles<false, TallTiles>(p);
    else lin1_swiglu_tiles<false, Short>(p);
  }
}
template <bool BWD, class Short>
constexpr size_t kLin1Lds = BWD ? Lin1Prog<BWD, Short>::kLds
                                : std::max(Lin1Prog<false, TallTiles>::kLds, Lin1Prog<false, Short>::kLds);
template <bool BWD, class Short>
__global__ __launch_bounds__(kThreads, 2) void lin1_swiglu_kernel(Lin1Args p) {
  const ClockTrace trace(p.clk);
  lin1_swiglu_by_table<BWD, Short>(p);
  trace.finish();
}
template <bool BWD, class Short>
int launch_lin1(const Lin1Args& a, hipStream_t st) {
  static LdsLimit lds;
  constexpr size_t bytes = kLin1Lds<BWD, Short>;
  if (!allow_lds(lin1_swiglu_kernel<BWD, Short>, bytes, lds)) return MOMOE_ERR_LAUNCH;
  lin1_swiglu_kernel<BWD, Short><<<persistent_grid(), kThreads, bytes, st>>>(a);
  return launch_status();
}
// Few tiles: NarrowTiles if the table holds as few as the launch was chosen for.  The SwiGLU backward
// writes twice as many partial row sums, each over 64 hidden columns: 1024 tokens over 32 experts,
// D = 1024, H = 512: 27.5 -> 21.6 us.
template <bool BWD>
__global__ __launch_bounds__(kThreads, 2) void lin1_swiglu_narrow_kernel(Lin1Args p) {
  // the backward's table has no taller tiles
  using Sched = std::conditional_t<BWD, TileSchedT<NarrowTiles::WROWS>, OneGeometrySched<NarrowTiles>>;
  constexpr int BNH = NarrowTiles::COLS / 2;
  const ClockTrace trace(p.clk);
  if (__builtin_expect(narrow_tiles_fit(p.table, (p.H + BNH - 1) / BNH), 1))
    lin1_swiglu_tiles<BWD, NarrowTiles, Sched>(p);
  else
    lin1_swiglu_by_table<BWD, StdTilesHalfParts>(p);
  trace.finish();
}
template <bool BWD>
int launch_lin1_narrow(const Lin1Args& a, hipStream_t st) {
  static LdsLimit lds;
  constexpr size_t bytes = std::max(Lin1Prog<BWD, NarrowTiles>::kLds, kLin1Lds<BWD, StdTilesHalfParts>);
  if (!allow_lds(lin1_swiglu_narrow_kernel<BWD>, bytes, lds)) return MOMOE_ERR_LAUNCH;
  lin1_swiglu_narrow_kernel<BWD><<<persistent_grid(), kThreads, bytes, st>>>(a);
  return launch_status();
}

// The same with dL/dh made on the way, for few tiles: u = G_y[idx] . Wl2^T contracts over D like a|b, for the same
// tokens, so both products share a main loop, and u of the tile's 64 hidden columns is rounded as momoe_dgrad_h would store it,
// but stays in registers.  A launch of few tiles is bound by what lies before its first and behind its last stage (5 us) and by the
// way of a stage from the L2, not by products: of two launches, the first with as many tiles as half of the second's, one is left, with
// 44 KiB a stage where each had 24, three stages (all that fit the LDS).  Two launches -> one, a step in us: 1024 tokens, D =
// 1024, H = 512, N = 32, K = 4 146 -> 140 (18.5 + 22.9 -> 33.7 of the GPU's); 700 of that kind, falling as rank^-1.8, 158 -> 152; 200, 2048, 768,
// 16, 2 182 -> 178; 3000, 256, 256, 16, 1 105 -> 102; 128, 128, 64, 8, 2, bound by the host, 96 -> 94; wide tiles: 1600, 1024, 512, 32, 4,
// rank^-0.5, 244 -> 234; 800, 2048, 1024, 16, 4 311 -> 304.  Below 3072 k-values: the longer a CU's share, the less the launch
// saved is of it.  H = 2048, N = 8, K = 4, 110 | 256 | 400 tokens, the last falling as rank^-0.5: D = 2592 236 -> 227 | 305 -> 295 | 436 ->
// 440, 2816 257 -> 252 | 326 -> 319 | 480 -> 481, 3040 279 -> 276 | 351 -> 345 | 508 -> 514; 400, 3040, 960, 16, 6 364 -> 361; from the line on
// D = 3072, 256 tokens 340 -> 333, 400 497 -> 502; 4096, 110 tokens 327 -> 329, 170 364 -> 359, 400 604 -> 609.  What loses there, and
// 1 % below (2048, 400 tokens 321 -> 324), are tiles a few too many for narrow ones: 144 wide ones leave half of the CUs
// idle in either form, which the host cannot know; other such loads gain (800, 2560, 1024, 16, 4, rank^-1.8 436 -> 416; 1500, 2816, 512, 32, 4
// 501 -> 478).  And up to one and a half row tiles per expert:
// 600, 2048, 768, 8, 4 (300 rows) 214 -> 206; past it 2048, 512, 256, 16, 4 126 -> 122 and 4000, 256, 128, 16, 2 114 -> 117, no more
// than the runs of one side differ by.
struct Lin1DhProg : Lin1Prog<true, NarrowTiles> {
  using Base = Lin1Prog<true, NarrowTiles>;
  using RowsOp = TwoRowsDma<NarrowTiles::AROWS>;
  using WeightOp = ColsAndRowsDma<NarrowTiles::COLS>;
  static_assert(WeightOp::ROWS == BNH, "the rows of Wl2 are those of the tile's hidden columns");
  using Ring = StageRing<RowsOp, WeightOp, 3>;
  static constexpr int NF = 3;  // column fragments: a, b, u
  __device__ __forceinline__ void setup(const TileCoord& t, const Prep& g, RowsOp& A, WeightOp& B) const {
    const int D = p.D, H = p.H, j0 = t.tn * BNH;
    A.init(p.x, p.gy, [&](int, int j) { return (uint32_t)g.tok[j] * (uint32_t)(2 * D); });
    B.t.init(p.w1 + (int64_t)t.expert * D * 2 * H, [&](int c) { return (c / BNH) * H + min(j0 + (c % BNH), H - 8); }, 2 * H);
    B.init_rows(p.w2 + (int64_t)t.expert * H * D, [&](int r) { return (uint32_t)min(j0 + r, H - 1) * (uint32_t)(2 * D); });
  }
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x16 (&acc)[NF][FM], const Prep& g, bf16* epi) const {
    epilogue_bwd(tc, acc, g, epi, [&](int i, bf16x4 (&uq)[4]) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        uq[q] = pack_bf16x4(acc[2][i][4 * q], acc[2][i][4 * q + 1], acc[2][i][4 * q + 2], acc[2][i][4 * q + 3]);
    });
  }
};
// Where the table holds more tiles than those, the tiles are wide ones, which have no registers for u.  It goes
// through memory there, but not past the workgroup: its 128 hidden columns of a row tile are a tile of either loop,
// dealt out alike, so a workgroup first makes u for all tiles that it will read it for.
__global__ __launch_bounds__(kThreads, 2) void lin1_dh_narrow_kernel(Lin1Args p) {
  const ClockTrace trace(p.clk);
  using Prog = Lin1DhProg;
  const int nb = (p.H + Prog::BNH - 1) / Prog::BNH;
  if (__builtin_expect(narrow_tiles_fit(p.table, nb), 1)) {
    typename Prog::Ring ring(dyn_lds());
    TileSchedT<NarrowTiles::WROWS> sched(p.table, nb, Prog::BM);
    const int wn = wave_id() % NarrowTiles::WCOLS;
    const int n_org[Prog::NF] = {wn * 32, Prog::BNH + wn * 32, wn * 32};
    Prog prog{{p, p.D / kBK, wn}};
    run_row_tiles<Prog::FM, Prog::NF>(prog, sched, ring, n_org);
  } else {
    using Wide = Lin1Prog<true, StdTilesHalfParts>;
    static_assert(Wide::BNH == NarrowTiles::COLS && Wide::BM == NarrowTiles::MAX_ROWS, "the same tiles");
    dgrad_h_tiles<NarrowTiles, TileSchedT<NarrowTiles::WROWS>>(
        DhArgs{p.gy, p.w2, p.idx, p.table, const_cast<bf16*>(p.u), p.D, p.H, nullptr}, Wide::BM);
    __syncthreads();  // u has been stored, the ring has been read
    lin1_swiglu_tiles<true, StdTilesHalfParts>(p);
  }
  trace.finish();
}
constexpr size_t kLin1DhLds =
    std::max({Lin1DhProg::Ring::BYTES, DhProg<NarrowTiles>::Ring::BYTES, Lin1Prog<true, StdTilesHalfParts>::kLds});

// The few-row tiles (FewRows): 32 `a` columns and their 32 `b` columns.
__global__ __launch_bounds__(kThreads, 2) void lin1_swiglu_few_rows_kernel(Lin1Args p) {
  constexpr int BNH = FewRows::G::COLS / 2;
  const ClockTrace trace(p.clk);
  bf16* lds = dyn_lds();
  const int first_tile = p.h == nullptr && p.ab_lo > 0 ? TileSched::expert_tile_of_row(p.table, p.ab_lo) : 0;
  FewRows::Sched sched(p.table, (p.H + BNH - 1) / BNH, first_tile);
  const int D = p.D, H = p.H;
  FewRows op;
  for (TileCoord left = sched.next(); left.valid; left = FewRows::following(sched, left)) {
    const TileCoord t = FewRows::piece(left);
    const FewRows::Tokens tokens(p.idx + t.row0, t.rows);
    const int j0 = t.tn * BNH;
    op.weights(p.w1 + (int64_t)t.expert * D * 2 * H, D,
               [&](int c) { return (c / BNH) * H + min(j0 + (c % BNH), H - 8); }, 2 * H);
    __builtin_amdgcn_s_barrier();  // the previous tile's partial sums have been read
    op.request_weights(lds, D);
    op.rows(p.x, FewRows::BK, D, [&](int, int piece) { return tokens.mine() * (uint32_t)(2 * D) + piece * 16; });
    f32x4 sum[FN];
    op.multiply(sum, lds, D, [] {});
    const int col = j0 + FewRows::column();
    const int64_t r = t.row0 + acc_row();
    if (FewRows::stores() && acc_row() < t.rows) {
      const f32x4 a = sum[0], b = sum[1];
      if (p.h)  // k-blocked: the tile's columns are one block
        store_bf16x4(p.h + ((int64_t)(j0 >> 5) * p.msum + r) * 32 + FewRows::column(), a[0] * b[0] * sigmoidf_fast(b[0]),
                     a[1] * b[1] * sigmoidf_fast(b[1]), a[2] * b[2] * sigmoidf_fast(b[2]), a[3] * b[3] * sigmoidf_fast(b[3]));
      if (p.ab && r >= p.ab_lo && r < p.ab_hi) {
        store_bf16x4(p.ab + r * 2 * H + col, a[0], a[1], a[2], a[3]);
        store_bf16x4(p.ab + r * 2 * H + H + col, b[0], b[1], b[2], b[3]);
      }
    }
    wait_lgkm0();
  }
  trace.finish();
}

struct Lin2Args {
  const bf16* h;
  const bf16* w2;
  const float* s;
  int64_t ssn, ssm;
  const int32_t* idx;
  const int32_t* table;
  bf16* ys;
  int D, H;
  int64_t msum;
  unsigned long long* clk;
};

struct Lin2Span {
  using G = WideSpan;
  static constexpr bool EXCHANGE = false;
  using Rows = SpanBlockedRows<256>;   // rows of h, k-blocked
  using Weights = SpanCols<>;
  using Ids = RowIds;     // tokens of the rows this wave holds in the accumulators
  using Late = RowScales; // their gate weights
  const Lin2Args& p;
  const int K, n_org;

  __device__ __forceinline__ explicit Lin2Span(const Lin2Args& p_)
      : p(p_), K(p_.H), n_org(wave_id() % G::WCOLS * (16 * G::FN)) {}
  __device__ __forceinline__ void gather(const TileCoord& t, Ids& g) const { g.gather(t, p.idx); }
  __device__ __forceinline__ void late(const TileCoord& t, const Ids& g, Late& s) const {
    s.load(t, g, p.s, p.ssn, p.ssm);
  }
  __device__ __forceinline__ void settle(Ids& g) const { g.settle(); }
  __device__ __forceinline__ void settle(Late& s) const { s.settle(); }
  __device__ __forceinline__ void setup(const TileCoord& t, const Ids&, Rows& A, Weights& W) const {
    const int D = p.D, d0 = t.tn * G::COLS;
    A.init(p.h, p.msum, t.row0, t.rows);
    W.init(p.w2 + (int64_t)t.expert * p.H * D, D, [&](int c) { return min(d0 + c, D - 8); });
  }
  template <int NA>
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x4 (&acc)[G::FN][NA], const Ids&, const Late& s,
                                           bf16* staging) const {
    const int lane = fresh_lane();
    store_rows(acc, staging, p.ys, (int64_t)tc.row0 + tc.mbase, tc.rows - tc.mbase, p.D, tc.tn * G::COLS + n_org, lane,
               [&](int i) { return s.of(i, lane); });
  }
};

__global__ __launch_bounds__(kSpanThreads, 1) void lin2_scale_kernel(Lin2Args p) {
  const ClockTrace trace(p.clk);
  run_span_tiles<Lin2Span>(p, (p.D + WideSpan::COLS - 1) / WideSpan::COLS, MOMOE_TILE_ROWS);
  trace.finish();
}

template <class G>
struct Lin2Prog {
  static constexpr int FM = G::FM, BN = G::COLS;
  static constexpr bool MAY_ONCE = G::MAY_ONCE;
  using HRowsOp = RBlockedDma<G::AROWS>;  // rows of h, k-blocked
  using WeightOp = TDmaT<BN, MAY_ONCE>;  // expert weights [k][col], k-strided
  using Ring = StageRing<HRowsOp, WeightOp, G::STAGES>;
  static constexpr size_t kLds = Ring::BYTES;
  struct Prep {
    int32_t tok[FM];  // tokens of the rows this lane holds in the accumulators
    float sv[FM];     // their gate weights
  };
  const Lin2Args& p;
  const int ktiles, wn;

  __device__ __forceinline__ void gather(const TileCoord& t, Prep& g) const {
#pragma unroll
    for (int i = 0; i < FM; ++i) g.tok[i] = p.idx[t.row0 + min(t.mbase + 32 * i + acc_row(), t.rows - 1)];
  }
  __device__ __forceinline__ void late(const TileCoord& t, Prep& g) const {
#pragma unroll
    for (int i = 0; i < FM; ++i) g.sv[i] = p.s[(int64_t)t.expert * p.ssn + (int64_t)g.tok[i] * p.ssm];
  }
  __device__ __forceinline__ void setup(const TileCoord& t, const Prep&, HRowsOp& A, WeightOp& B) const {
    const int D = p.D, H = p.H;
    const bf16* w = p.w2 + (int64_t)t.expert * H * D;
    const int d0 = t.tn * BN;
    A.init(p.h, p.msum, t.row0, t.rows);
    B.init(w, [&](int c) { return min(d0 + c, D - 8); }, D);
    if (MAY_ONCE) B.once = t.alone;
  }
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x16 (&acc)[FN][FM], const Prep& g, bf16* epi) const {
    const int D = p.D;
    const RowStager<2> stager(epi);
    const int d0 = tc.tn * BN + wn * 64;  // first output column of this wave
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i >= tc.na) break;
      const float sv = g.sv[i];
#pragma unroll
      for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          stager.put(f, q, pack_bf16x4(acc[f][i][4 * q] * sv, acc[f][i][4 * q + 1] * sv,
                                       acc[f][i][4 * q + 2] * sv, acc[f][i][4 * q + 3] * sv));
      stager.flush([&](int row, int col) -> bf16* {
        const int rl = (tc.mbase + 32 * i) + row;
        if (rl >= tc.rows || d0 + col >= D) return nullptr;
        return p.ys + ((int64_t)tc.row0 + rl) * D + d0 + col;
      });
    }
  }
};

template <class G, class Sched = TileSched>
__device__ __forceinline__ void lin2_scale_tiles(const Lin2Args& p) {
  using Prog = Lin2Prog<G>;
  typename Prog::Ring ring(dyn_lds());
  Sched sched(p.table, (p.D + G::COLS - 1) / G::COLS, MOMOE_TILE_ROWS);
  const int wn = wave_id() % G::WCOLS;
  const int n_org[FN] = {wn * 64, wn * 64 + 32};
  Prog prog{p, p.H / kBK, wn};
  run_row_tiles<Prog::FM, FN>(prog, sched, ring, n_org);
}

template <class Short>
__device__ __forceinline__ void lin2_scale_by_table(const Lin2Args& p) {
  if (TileSched::tile_rows_of(p.table) > Short::MAX_ROWS) lin2_scale_tiles<TallTiles>(p);
  else lin2_scale_tiles<Short>(p);
}
template <class Short>
constexpr size_t kLin2Lds = std::max(Lin2Prog<TallTiles>::kLds, Lin2Prog<Short>::kLds);
template <class Short>
__global__ __launch_bounds__(kThreads, 2) void lin2_scale_once_kernel(Lin2Args p) {
  const ClockTrace trace(p.clk);
  lin2_scale_by_table<Short>(p);
  trace.finish();
}
template <class Short>
int launch_lin2(const Lin2Args& a, hipStream_t st) {
  static LdsLimit lds;
  constexpr size_t bytes = kLin2Lds<Short>;
  if (!allow_lds(lin2_scale_once_kernel<Short>, bytes, lds)) return MOMOE_ERR_LAUNCH;
  lin2_scale_once_kernel<Short><<<persistent_grid(), kThreads, bytes, st>>>(a);
  return launch_status();
}
__global__ __launch_bounds__(kThreads, 2) void lin2_scale_narrow_kernel(Lin2Args p) {
  const ClockTrace trace(p.clk);
  if (__builtin_expect(narrow_tiles_fit(p.table, (p.D + NarrowTiles::COLS - 1) / NarrowTiles::COLS), 1))
    lin2_scale_tiles<NarrowTiles, OneGeometrySched<NarrowTiles>>(p);
  else
    lin2_scale_by_table<StdTiles>(p);
  trace.finish();
}
constexpr size_t kLin2NarrowLds = std::max(Lin2Prog<NarrowTiles>::kLds, kLin2Lds<StdTiles>);

__global__ __launch_bounds__(kThreads, 2) void lin2_scale_few_rows_kernel(Lin2Args p) {
  const ClockTrace trace(p.clk);
  bf16* lds = dyn_lds();
  FewRows::Sched sched(p.table, (p.D + FewRows::G::COLS - 1) / FewRows::G::COLS, 0);
  const int D = p.D, H = p.H;
  FewRows op;
  for (TileCoord left = sched.next(); left.valid; left = FewRows::following(sched, left)) {
    const TileCoord t = FewRows::piece(left);
    // The gate weights of the rows come through the scalar unit, too: a chain of two loads, each waited for a step later; most
    // tiles have no more rows than the first of them
    constexpr int kAtOnce = 8;
    const int32_t* const idx = p.idx + t.row0;
    const float* const s = p.s + (int64_t)t.expert * p.ssn;
    int32_t tok[kAtOnce];
    float sv[kAtOnce], mine = 0.0f;
    auto load_tokens = [&](int r0) {
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i) tok[i] = load_uniform(idx + min(r0 + i, t.rows - 1));
    };
    auto load_gate_weights = [&] {
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i) sv[i] = load_uniform(s + (int64_t)tok[i] * p.ssm);
    };
    auto keep_mine = [&](int r0) {
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i) mine = acc_row() == r0 + i ? sv[i] : mine;
    };
    load_tokens(0);
    const int d0 = t.tn * FewRows::G::COLS;
    op.weights(p.w2 + (int64_t)t.expert * H * D, H, [&](int c) { return min(d0 + c, D - 8); }, D);
    __builtin_amdgcn_s_barrier();  // the previous tile's partial sums have been read
    op.request_weights(lds, H);
    // h is k-blocked: a stage is four blocks of 32 k-values
    const uint32_t block = (uint32_t)p.msum * (kBK * 2);
    op.rows(p.h + (int64_t)t.row0 * kBK, 4 * p.msum * kBK, H, [&](int row, int piece) {
      return (uint32_t)min(row, t.rows - 1) * (kBK * 2) + (piece >> 2) * block + (piece & 3) * 16;
    });
    f32x4 sum[FN];
    op.multiply(sum, lds, H, [&] {
      if (FewRows::stores())
        for (int r0 = kAtOnce; r0 < t.rows; r0 += kAtOnce) {
          load_gate_weights();
          keep_mine(r0 - kAtOnce);
          load_tokens(r0);
        }
      load_gate_weights();
    });
    keep_mine((t.rows - 1) / kAtOnce * kAtOnce);
    if (FewRows::stores() && acc_row() < t.rows) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = d0 + 32 * j + FewRows::column();
        if (col < D)
          store_bf16x4(p.ys + (int64_t)(t.row0 + acc_row()) * D + col, sum[j][0] * mine, sum[j][1] * mine, sum[j][2] * mine,
                       sum[j][3] * mine);
      }
    }
    wait_lgkm0();
  }
  trace.finish();
}

// out[m] = sum_k rows[inv[m,k]]: one workgroup per token, 16-byte loads, fp32 accumulate.
// The row numbers and then the rows are fetched 8 at a time with unconditional loads (a missing
// pair, inv = -1, is pointed at row 0 and left out of the sum): loads under a branch would be
// waited for one by one.  Bound by HBM; every row is read once and not again.  ONCE
// (kBeyondCache): 65536 rows of 2048 (302 MB in and out) 54.2 -> 48.2 us = 6.3 TB/s.
template <bool ONCE>
__global__ __launch_bounds__(256) void combine_kernel(const bf16* __restrict__ rows,
                                                      const int32_t* __restrict__ inv,
                                                      bf16* __restrict__ out, int D, int K,
                                                      int64_t msum) {
  const int64_t m = blockIdx.x;
  for (int c = threadIdx.x; c < D / 8; c += blockDim.x) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k0 = 0; k0 < K; k0 += 8) {
      int32_t r[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = inv[m * K + min(k0 + j, K - 1)];
      bf16x8 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool ok = k0 + j < K && (uint32_t)r[j] < (uint64_t)msum;
        v[j] = load_maybe_once<ONCE>((const bf16x8*)(rows + (int64_t)(ok ? r[j] : 0) * D + c * 8));
        r[j] = ok ? 1 : 0;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += r[j] ? (float)v[j][e] : 0.0f;
    }
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)acc[e];
    *(bf16x8*)(out + m * D + c * 8) = o;
  }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

inline int check_dims(int64_t M, int64_t D, int64_t H, int64_t N, int64_t Msum) {
  if (M <= 0 || D <= 0 || H <= 0 || N <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  if (D % kBK != 0 || H % kBK != 0) return MOMOE_ERR_UNSUPPORTED;
  // per-lane source offsets are 32-bit byte offsets from x / from an expert's weights
  if (Msum >= (1ll << 31) || M * D * 2 >= (1ll << 32) || D * H * 4 >= (1ll << 32))
    return MOMOE_ERR_UNSUPPORTED;
  return MOMOE_OK;
}

}  // namespace
}  // namespace momoe

using namespace momoe;

extern "C" int momoe_lin1_swiglu_fwd(const void* x_MD, const void* Wl1_ND2H,
                                     const int32_t* idx_Msum, const int32_t* tile_table,
                                     void* h_blocked, void* ab_rows, int64_t ab_row_lo,
                                     int64_t ab_row_hi, int64_t M, int64_t D, int64_t H,
                                     int64_t N, int64_t Msum, void* stream) {
  if (!x_MD || !Wl1_ND2H || !idx_Msum || !tile_table || (!h_blocked && !ab_rows))
    return MOMOE_ERR_BAD_ARG;
  if (!aligned16(x_MD) || !aligned16(Wl1_ND2H) || ((uintptr_t)h_blocked & 15) ||
      ((uintptr_t)ab_rows & 15))
    return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  Lin1Args a{(const bf16*)x_MD, (const bf16*)Wl1_ND2H, idx_Msum, tile_table, (bf16*)h_blocked,
             (bf16*)ab_rows, ab_row_lo, ab_row_hi, (int)D, (int)H,
             nullptr, nullptr, 0, 0, nullptr, nullptr, 0, nullptr, Msum, clock_trace_buffer()};
  if (takes_few_rows_tiles(M, Msum, N, 2 * H)) {
    static LdsLimit few;
    if (!allow_lds(lin1_swiglu_few_rows_kernel, FewRows::BYTES, few)) return MOMOE_ERR_LAUNCH;
    lin1_swiglu_few_rows_kernel<<<persistent_grid(), kThreads, FewRows::BYTES, (hipStream_t)stream>>>(a);
    return launch_status();
  }
  if (takes_span_tiles(Msum, N, 2 * H, D)) {
    static LdsLimit span;
    return launch_span(lin1_swiglu_fwd_kernel, a, span, (hipStream_t)stream);
  }
  if (!takes_narrow_tiles(Msum, N, 2 * H) && weights_read_once(Msum, N, 4 * N * D * H))
    return launch_lin1<false, OnceTiles>(a, (hipStream_t)stream);
  return launch_lin1_narrow<false>(a, (hipStream_t)stream);
}

extern "C" int momoe_gemm_tile_rows(int64_t Msum, int64_t N, int64_t cols, int64_t contraction) {
  if (Msum <= 0 || N <= 0 || cols <= 0 || contraction <= 0) return 0;
  return takes_span_tiles(Msum, N, cols, contraction) ? MOMOE_RECOMPUTE_TILE_ROWS : 0;
}

extern "C" int momoe_recompute_stage_k(int64_t Msum, int64_t N, int64_t D, int64_t H) {
  if (Msum <= 0 || N <= 0 || D <= 0 || H <= 0) return 0;
  return takes_span_recompute(Msum, N, H, D) ? kSpan : kBK;
}

extern "C" int64_t momoe_gs_parts(int64_t H, int64_t N, int64_t Msum) {
  if (H <= 0 || N <= 0 || Msum <= 0) return -1;
  return cdiv64(H, takes_narrow_tiles(Msum, N, 2 * H) ? MOMOE_GS_BLOCK / 2 : MOMOE_GS_BLOCK);
}

extern "C" int momoe_lin1_swiglu_bwd(const void* x_MD, const void* Wl1_ND2H,
                                     const int32_t* idx_Msum, const int32_t* tile_table,
                                     const void* u_MsumH, const float* s_NM, int64_t s_stride_n,
                                     int64_t s_stride_m, int64_t row_lo, void* gz_blocked,
                                     void* hsT_GH32, int64_t ld_hsT, float* gs_part, int64_t M,
                                     int64_t D, int64_t H, int64_t N, int64_t Msum, void* stream) {
  return momoe_lin1_swiglu_bwd_parts(x_MD, Wl1_ND2H, idx_Msum, tile_table, u_MsumH, s_NM, s_stride_n,
                                     s_stride_m, row_lo, gz_blocked, hsT_GH32, ld_hsT, gs_part,
                                     cdiv64(std::max<int64_t>(H, 0), MOMOE_GS_BLOCK), M, D, H, N, Msum, stream);
}

extern "C" int momoe_lin1_swiglu_bwd_parts(const void* x_MD, const void* Wl1_ND2H,
                                           const int32_t* idx_Msum, const int32_t* tile_table,
                                           const void* u_MsumH, const float* s_NM, int64_t s_stride_n,
                                           int64_t s_stride_m, int64_t row_lo, void* gz_blocked,
                                           void* hsT_GH32, int64_t ld_hsT, float* gs_part,
                                           int64_t nparts, int64_t M, int64_t D, int64_t H, int64_t N,
                                           int64_t Msum, void* stream) {
  if (!x_MD || !Wl1_ND2H || !idx_Msum || !tile_table || !u_MsumH || !s_NM || !gz_blocked ||
      !hsT_GH32 || !gs_part)
    return MOMOE_ERR_BAD_ARG;
  if (row_lo < 0 || row_lo > Msum) return MOMOE_ERR_BAD_ARG;
  if (!aligned16(x_MD) || !aligned16(Wl1_ND2H) || ((uintptr_t)u_MsumH & 7) ||
      !aligned16(gz_blocked) || !aligned16(hsT_GH32))
    return MOMOE_ERR_BAD_ARG;
  if (ld_hsT < H || ld_hsT % 8 != 0) return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  // parts of 128 hidden columns, or of 64 where the launch can write those
  const bool narrow = nparts != cdiv64(H, MOMOE_GS_BLOCK) && takes_narrow_tiles(Msum, N, 2 * H);
  if (nparts != cdiv64(H, narrow ? MOMOE_GS_BLOCK / 2 : MOMOE_GS_BLOCK)) return MOMOE_ERR_BAD_ARG;
  if (row_lo == Msum) return MOMOE_OK;
  Lin1Args a{(const bf16*)x_MD, (const bf16*)Wl1_ND2H, idx_Msum, tile_table, nullptr, nullptr,
             row_lo, Msum, (int)D, (int)H, (const bf16*)u_MsumH, s_NM, s_stride_n, s_stride_m,
             (bf16*)gz_blocked, (bf16*)hsT_GH32, ld_hsT, gs_part, Msum, clock_trace_buffer()};
  if (narrow) return launch_lin1_narrow<true>(a, (hipStream_t)stream);
  if (takes_span_recompute(Msum, N, H, D)) {
    static LdsLimit span;
    return launch_span(lin1_swiglu_bwd_kernel, a, span, (hipStream_t)stream);
  }
  return launch_lin1<true, StdTiles>(a, (hipStream_t)stream);
}

extern "C" int momoe_dgrad_h_lin1_bwd_fits(int64_t M, int64_t D, int64_t H, int64_t N, int64_t Msum) {
  return check_dims(M, D, H, N, Msum) == MOMOE_OK && takes_narrow_tiles(Msum, N, 2 * H) && D < 3072 &&
         2 * Msum <= 3 * N * StdTiles::MAX_ROWS;
}

extern "C" int momoe_dgrad_h_lin1_bwd(const void* Gy_MD, const void* Wl2_NHD, const void* x_MD, const void* Wl1_ND2H,
                                      const int32_t* idx_Msum, const int32_t* tile_table, const float* s_NM, int64_t s_stride_n,
                                      int64_t s_stride_m, void* u_MsumH, void* gz_blocked, void* hsT_GH32, int64_t ld_hsT,
                                      float* gs_part, int64_t nparts, int64_t M, int64_t D, int64_t H, int64_t N, int64_t Msum,
                                      void* stream) {
  if (!Gy_MD || !Wl2_NHD || !x_MD || !Wl1_ND2H || !idx_Msum || !tile_table || !s_NM || !u_MsumH || !gz_blocked || !hsT_GH32 ||
      !gs_part)
    return MOMOE_ERR_BAD_ARG;
  for (const void* q : {Gy_MD, Wl2_NHD, x_MD, Wl1_ND2H, (const void*)u_MsumH, (const void*)gz_blocked, (const void*)hsT_GH32})
    if (!aligned16(q)) return MOMOE_ERR_BAD_ARG;
  if (ld_hsT < H || ld_hsT % 8 != 0) return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  if (!momoe_dgrad_h_lin1_bwd_fits(M, D, H, N, Msum)) return MOMOE_ERR_UNSUPPORTED;
  if (nparts != cdiv64(H, MOMOE_GS_BLOCK / 2)) return MOMOE_ERR_BAD_ARG;
  const Lin1Args a{(const bf16*)x_MD, (const bf16*)Wl1_ND2H, idx_Msum, tile_table, nullptr, nullptr,
                   0, Msum, (int)D, (int)H, (const bf16*)u_MsumH, s_NM, s_stride_n, s_stride_m,
                   (bf16*)gz_blocked, (bf16*)hsT_GH32, ld_hsT, gs_part, Msum, clock_trace_buffer(),
                   (const bf16*)Gy_MD, (const bf16*)Wl2_NHD};
  static LdsLimit lds;
  if (!allow_lds(lin1_dh_narrow_kernel, kLin1DhLds, lds)) return MOMOE_ERR_LAUNCH;
  lin1_dh_narrow_kernel<<<persistent_grid(), kThreads, kLin1DhLds, (hipStream_t)stream>>>(a);
  return launch_status();
}

extern "C" int momoe_lin2_scale_fwd(const void* h_blocked, const void* Wl2_NHD, const float* s_NM,
                                    int64_t s_stride_n, int64_t s_stride_m,
                                    const int32_t* idx_Msum, const int32_t* tile_table,
                                    void* ys_MsumD, int64_t M, int64_t D, int64_t H, int64_t N,
                                    int64_t Msum, void* stream) {
  if (!h_blocked || !Wl2_NHD || !s_NM || !idx_Msum || !tile_table || !ys_MsumD)
    return MOMOE_ERR_BAD_ARG;
  if (!aligned16(h_blocked) || !aligned16(Wl2_NHD) || ((uintptr_t)ys_MsumD & 7))
    return MOMOE_ERR_BAD_ARG;
  const int st = check_dims(M, D, H, N, Msum);
  if (st != MOMOE_OK) return st;
  Lin2Args a{(const bf16*)h_blocked, (const bf16*)Wl2_NHD, s_NM, s_stride_n, s_stride_m,
             idx_Msum, tile_table, (bf16*)ys_MsumD, (int)D, (int)H, Msum, clock_trace_buffer()};
  if (takes_few_rows_tiles(M, Msum, N, D)) {
    static LdsLimit few;
    if (!allow_lds(lin2_scale_few_rows_kernel, FewRows::BYTES, few)) return MOMOE_ERR_LAUNCH;
    lin2_scale_few_rows_kernel<<<persistent_grid(), kThreads, FewRows::BYTES, (hipStream_t)stream>>>(a);
    return launch_status();
  }
  if (takes_span_tiles(Msum, N, D, H)) {
    static LdsLimit span;
    return launch_span(lin2_scale_kernel, a, span, (hipStream_t)stream);
  }
  if (!takes_narrow_tiles(Msum, N, D) && weights_read_once(Msum, N, 2 * N * D * H))
    return launch_lin2<OnceTiles>(a, (hipStream_t)stream);
  static LdsLimit narrow;
  if (!allow_lds(lin2_scale_narrow_kernel, kLin2NarrowLds, narrow)) return MOMOE_ERR_LAUNCH;
  lin2_scale_narrow_kernel<<<persistent_grid(), kThreads, kLin2NarrowLds, (hipStream_t)stream>>>(a);
  return launch_status();
}

extern "C" int momoe_combine(const void* rows_MsumD, const int32_t* inv_MK, void* out_MD,
                             int64_t M, int64_t D, int64_t K, int64_t Msum, void* stream) {
  if (!rows_MsumD || !inv_MK || !out_MD) return MOMOE_ERR_BAD_ARG;
  if (M <= 0 || D <= 0 || K <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  if (D % 8 != 0 || M >= (1ll << 31) || Msum >= (1ll << 31)) return MOMOE_ERR_UNSUPPORTED;
  if (!aligned16(rows_MsumD) || !aligned16(out_MD)) return MOMOE_ERR_BAD_ARG;
  auto kernel = Msum * D * 2 >= kBeyondCache ? combine_kernel<true> : combine_kernel<false>;
  kernel<<<(unsigned)M, 256, 0, (hipStream_t)stream>>>(
      (const bf16*)rows_MsumD, inv_MK, (bf16*)out_MD, (int)D, (int)K, Msum);
  return launch_status();
}
