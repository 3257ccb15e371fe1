// dL/dx in sorted order in the loop of gemm_tile.hpp: a launch of its own (experts_bwd.hip), and a part of the launch that
// ends the backward of a small call (wgrad.hip).
#pragma once
#include <algorithm>

#include "gemm_tile.hpp"

namespace momoe {
namespace {

struct DxArgs {
  const bf16* gz;
  const bf16* w1;
  const int32_t* table;
  bf16* gxs;
  int D, H;
  int64_t msum;
  unsigned long long* clk;
};

// gxs = gz . Wl1^T: contraction over the 2H contiguous columns of both operands.
template <class G>
struct DxProg {
  static constexpr int FM = G::FM, BN = G::COLS;
  static constexpr bool MAY_ONCE = false;
  using BlockedA = RBlockedDma<G::AROWS>;  // sorted rows of the k-blocked gz
  using RowsB = RDma<BN>;                  // weight rows, k-contiguous
  using Ring = StageRing<BlockedA, RowsB, G::STAGES>;
  struct Prep {};
  const DxArgs& p;
  const int ktiles, wn;

  __device__ __forceinline__ void gather(const TileCoord&, Prep&) const {}
  __device__ __forceinline__ void late(const TileCoord&, Prep&) const {}
  __device__ __forceinline__ void setup(const TileCoord& t, const Prep&, BlockedA& A, RowsB& B) const {
    const int D = p.D, H2 = 2 * p.H;
    const bf16* w = p.w1 + (int64_t)t.expert * D * H2;
    const int d0 = t.tn * BN;
    A.init(p.gz, p.msum, t.row0, t.rows);
    B.init(w, [&](int r, int) { return (uint32_t)min(d0 + r, D - 1) * (uint32_t)(2 * H2); });
  }
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x16 (&acc)[2][FM], const Prep&, bf16* epi) const {
    const int D = p.D;
    const RowStager<2> stager(epi);
    const int d0 = tc.tn * BN + wn * 64;  // first output column of this wave
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i >= tc.na) break;
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          stager.put(f, q, pack_bf16x4(acc[f][i][4 * q], acc[f][i][4 * q + 1],
                                       acc[f][i][4 * q + 2], acc[f][i][4 * q + 3]));
      stager.flush([&](int row, int col) -> bf16* {
        const int rl = (tc.mbase + 32 * i) + row;
        if (rl >= tc.rows || d0 + col >= D) return nullptr;
        return p.gxs + ((int64_t)tc.row0 + rl) * D + d0 + col;
      });
    }
  }
};

template <class G, class Sched = TileSched>
__device__ __forceinline__ void dgrad_x_tiles(const DxArgs& p) {
  using Prog = DxProg<G>;
  typename Prog::Ring ring(dyn_lds());
  Sched sched(p.table, (p.D + G::COLS - 1) / G::COLS, MOMOE_TILE_ROWS);
  const int wn = wave_id() % G::WCOLS;
  const int n_org[2] = {wn * 64, wn * 64 + 32};
  Prog prog{p, (2 * p.H) / kBK, wn};
  run_row_tiles<Prog::FM, 2>(prog, sched, ring, n_org);
}

__device__ __forceinline__ void dgrad_x_by_table(const DxArgs& p) {
  if (TileSched::tile_rows_of(p.table) > StdTiles::MAX_ROWS) dgrad_x_tiles<TallTiles>(p);
  else dgrad_x_tiles<StdTiles>(p);
}
// Narrow tiles, or wide ones where the table has too many for those
__device__ __forceinline__ void dgrad_x_short(const DxArgs& p) {
  const ClockTrace trace(p.clk);
  if (__builtin_expect(narrow_tiles_fit(p.table, (p.D + NarrowTiles::COLS - 1) / NarrowTiles::COLS), 1))
    dgrad_x_tiles<NarrowTiles, OneGeometrySched<NarrowTiles>>(p);
  else
    dgrad_x_by_table(p);
  trace.finish();
}
constexpr size_t kDxLds = std::max(DxProg<TallTiles>::Ring::BYTES, DxProg<StdTiles>::Ring::BYTES);
constexpr size_t kDxNarrowLds = std::max(DxProg<NarrowTiles>::Ring::BYTES, kDxLds);

}  // namespace
}  // namespace momoe
