// dL/dh before the gate weight, in sorted order, in the loop of gemm_tile.hpp: a launch of its own (experts_bwd.hip), and part
// of the launch that makes it on the way to the SwiGLU backward (experts_fwd.hip).
#pragma once
#include "gemm_tile.hpp"

namespace momoe {
namespace {

struct DhArgs {
  const bf16* gy;
  const bf16* w2;
  const int32_t* idx;
  const int32_t* table;
  bf16* u;
  int D, H;
  unsigned long long* clk;
};

// u = G_y[idx] . Wl2^T is an "NT" GEMM: both operands are k-contiguous (k = D).
template <class G>
struct DhProg {
  static constexpr int FM = G::FM, BN = G::COLS;
  static constexpr bool MAY_ONCE = false;
  using RowsA = RDma<G::AROWS>;  // gathered token rows, k-contiguous
  using RowsB = RDma<BN>;        // weight rows, k-contiguous (an "NT" GEMM)
  using Ring = StageRing<RowsA, RowsB, G::STAGES>;  // its idle buffer is the store staging
  struct Prep {
    int32_t tok[RowsA::NCH];  // tokens of the rows this lane fetches
  };
  const DhArgs& p;
  const int ktiles, wn;

  __device__ __forceinline__ void gather(const TileCoord& t, Prep& g) const {
#pragma unroll
    for (int j = 0; j < RowsA::NCH; ++j) g.tok[j] = p.idx[t.row0 + min(RowsA::row_of(j), t.rows - 1)];
  }
  __device__ __forceinline__ void late(const TileCoord&, Prep&) const {}
  __device__ __forceinline__ void setup(const TileCoord& t, const Prep& g, RowsA& A, RowsB& B) const {
    const int D = p.D, H = p.H;
    const bf16* w = p.w2 + (int64_t)t.expert * H * D;
    const int n0 = t.tn * BN;
    A.init(p.gy, [&](int, int j) { return (uint32_t)g.tok[j] * (uint32_t)(2 * D); });
    B.init(w, [&](int r, int) { return (uint32_t)min(n0 + r, H - 1) * (uint32_t)(2 * D); });
  }
  __device__ __forceinline__ void epilogue(const TileCoord& tc, f32x16 (&acc)[2][FM], const Prep&, bf16* epi) const {
    const int H = p.H;
    const RowStager<2> stager(epi);
    const int n0 = tc.tn * BN + wn * 64;  // first hidden column of this wave
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
        if (rl >= tc.rows || n0 + col >= H) return nullptr;
        return p.u + ((int64_t)tc.row0 + rl) * H + n0 + col;
      });
    }
  }
};

template <class G, class Sched = TileSched>
__device__ __forceinline__ void dgrad_h_tiles(const DhArgs& p, int max_tile_rows = MOMOE_TILE_ROWS) {
  using Prog = DhProg<G>;
  typename Prog::Ring ring(dyn_lds());
  Sched sched(p.table, (p.H + G::COLS - 1) / G::COLS, max_tile_rows);
  const int wn = wave_id() % G::WCOLS;
  const int n_org[2] = {wn * 64, wn * 64 + 32};
  Prog prog{p, p.D / kBK, wn};
  run_row_tiles<Prog::FM, 2>(prog, sched, ring, n_org);
}

}  // namespace
}  // namespace momoe
