// Weight-gradient grouped GEMM: GW[i] = A_i^T . B_i, contracting over the sorted
// rows of expert i.  An operand is handed over in one of three layouts:
//   rows        [row][feature] (optionally gathered through an index: x and G_y are never
//               materialised in sorted order).  The contraction index is the slow one, so its
//               fragments come through the LDS transpose read, at half the rate of a plain read.
//   transposed  [padded sorted row / 32][feature][32]: the producing kernel wrote the matrix in
//               groups of 32 rows, feature-major inside a group (hs), each expert's rows starting
//               at a multiple of 32 and zero-filled up to the next multiple of 32.  The
//               contraction index is the fast one: plain 16-byte fragment reads, and a stage is
//               one contiguous 16 KiB block in memory.
//   k-blocked   (B only) blocks of 32 features, [feature / 32][row][32]: as rows for the fragments.
// Two loops: that of gemm_span.hpp, 64 rows a stage, and for few rows per expert that of gemm_tile.hpp
// (takes_span_loop).  The k-values past the expert's last row are zeroed in registers on the M side.
#include <algorithm>

#include "dgrad_x.hpp"
#include "gemm_span.hpp"
#include "gs_tokens.hpp"

namespace momoe {
namespace {

constexpr int BX = 256;  // output rows per tile (features of A)
constexpr int BY = 256;  // output columns per tile (features of B)
constexpr int kMaxWgradExperts = 4096;  // 20 bytes of prefix sums per expert fit the stage rings
constexpr int kMaxWorkgroups = 256;       // the workspace query assumes no more persistent workgroups
constexpr int kSplitsPerWorkgroup = 8;  // large experts are cut into pieces of 1/8 .. 1/4 of a
                                        // workgroup's share of the launch
static_assert(BX * BY * 4 == MOMOE_WGRAD_PARTIAL_BYTES, "size of one fp32 partial tile");

struct WgradArgs {
  const bf16* a;
  int64_t lda;
  const int32_t* ga;
  const bf16* b;
  int64_t ldb;
  const int32_t* gb;
  const int32_t* cumsums;
  bf16* gw;
  float* ws;      // fp32 partial tiles of the experts that are cut along their rows
  int kc;         // experts of at least 2*kc k-stages are cut into pieces of kc .. 2*kc stages
  int N, X, Y;
  int tiles_x, tiles_y;
  int msum;       // rows of the sorted matrices: row counts are clamped to it
  unsigned long long* clk;
};

// A work item's rows: sorted rows [rb, re) and its first padded row; all zero where it has none
struct Span {
  int rb, re, prow;
  __device__ __forceinline__ void forget_if_empty() {
    if (re <= rb) rb = re = prow = 0;
  }
  __device__ __forceinline__ int stages() const { return max(2, (re - rb + kSpan - 1) / kSpan); }
};

struct WTile {
  int expert, q;  // q-th output tile of the expert
  int x0, y0;     // where that is
  Span rows;  // this work item contracts over
  int slot;   // partial tile to write, or -1: the item covers the whole expert and stores bf16
  int valid;
};

constexpr int kBandTiles = 4;
// Estimated time of an item in units of 32 rows of its main loop; every item has its stores.  In the loop of
// gemm_span.hpp it has two stages of 64 at least, and items without rows are no part of it (they cost nothing here)
template <int THREADS>
__device__ __forceinline__ int item_cost(int ks) {
  constexpr int kStoreCost = 4;
  if (THREADS != kSpanThreads) return ks + kStoreCost;
  return ks > 0 ? max(4, ks + (ks & 1)) + kStoreCost : 0;
}
constexpr int kMinChunk = 64;     // an expert is never cut into pieces of fewer k-stages
// momoe_backward_tail_fits: what gz, gxs and s*h may take together, a bound on memory: one launch was the faster one in each of
// 37 calls of 0.2 to 63 MiB and up to 4095 tokens, with even loads, loads that fall as rank^-0.5 and rank^-1.8 and shared experts.  A
// step near the line, us, four launches -> one: 4095 tokens, D = 512, H = 2048, N = 64, K = 1 (60 MiB) rank^-1.8 361 -> 282; 4095,
// 4096, 1024, 16, 1 (57) even 626 -> 599, rank^-1.8 766 -> 645; 700, 2048, 768, 128, 8 (52) 912 -> 893, 677 -> 641; 1500, 1024, 512,
// 64, 8 (61), two of them shared, 407 -> 356; 300, 4096, 1408, 128, 8 (49) rank^-0.5 3040 -> 2955.
constexpr int64_t kTailBytes = 64 << 20;

// How one expert's rows are dealt out: `splits` equal pieces of `chunk` k-stages (the last
// may be shorter).  An expert is cut once it holds at least 2*kc stages, so a piece has
// between kc and 2*kc stages.
struct ExpertPlan {
  int ks, splits, chunk;
};
__device__ __forceinline__ ExpertPlan plan_expert(int rows, int kc) {
  ExpertPlan e;
  e.ks = (rows + kBK - 1) / kBK;
  e.splits = max(1, e.ks / kc);
  e.chunk = (e.ks + e.splits - 1) / e.splits;
  return e;
}

// Prefix sums over the experts, kept in LDS while the work is dealt out (they overlay the
// stage ring).  A work item is one output tile of one piece of one expert; inside an expert
// the items run piece by piece, tile by tile.
struct Plan {
  int64_t* cost;    // [N+1] estimated cost of the items of the experts before e
  int32_t* items;   // [N+1] items of the experts before e
  int32_t* slots;   // [N+1] partial tiles of the experts before e (cut experts only)
  int32_t* ctiles;  // [N+1] output tiles of the cut experts before e
  int kc;
};

template <int THREADS>
__device__ __forceinline__ Plan build_plan(const WgradArgs& p, int tpe) {
  Plan pl;
  pl.cost = (int64_t*)dyn_lds();
  pl.items = (int32_t*)(pl.cost + p.N + 1);
  pl.slots = pl.items + p.N + 1;
  pl.ctiles = pl.slots + p.N + 1;
  int64_t* wt = (int64_t*)(((uintptr_t)(pl.ctiles + p.N + 1) + 7) & ~(uintptr_t)7);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per = (p.N + THREADS - 1) / THREADS;  // experts per thread, contiguous
  const int e0 = min((int)threadIdx.x * per, p.N), e1 = min(e0 + per, p.N);

  pl.kc = p.kc;

  // exclusive scans of cost / items / slots / cut tiles over the experts
  int64_t c = 0;
  int32_t n = 0, sl = 0, ct = 0;
  for (int e = e0; e < e1; ++e) {
    const ExpertPlan ep = plan_expert(min(p.cumsums[e + 1], p.msum) - min(p.cumsums[e], p.msum), pl.kc);
    const int ne = tpe * ep.splits;
    c += (int64_t)ne * item_cost<THREADS>(ep.chunk);
    n += ne;
    if (ep.splits > 1) sl += ne, ct += tpe;
  }
  int64_t ic = c;
  int32_t in = n, isl = sl, ict = ct;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t vc = __shfl_up(ic, o);
    const int32_t vn = __shfl_up(in, o), vs = __shfl_up(isl, o), vt = __shfl_up(ict, o);
    if (lane >= o) ic += vc, in += vn, isl += vs, ict += vt;
  }
  if (lane == 63) {  // per wave: cost, items, slots, cut tiles
    wt[4 * wave] = ic;
    wt[4 * wave + 1] = in;
    wt[4 * wave + 2] = isl;
    wt[4 * wave + 3] = ict;
  }
  __syncthreads();
  int64_t bc = 0;
  int32_t bn = 0, bs = 0, bt = 0;
  for (int w = 0; w < wave; ++w) {
    bc += wt[4 * w];
    bn += (int32_t)wt[4 * w + 1];
    bs += (int32_t)wt[4 * w + 2];
    bt += (int32_t)wt[4 * w + 3];
  }
  bc += ic - c, bn += in - n, bs += isl - sl, bt += ict - ct;
  for (int e = e0; e < e1; ++e) {
    pl.cost[e] = bc, pl.items[e] = bn, pl.slots[e] = bs, pl.ctiles[e] = bt;
    const ExpertPlan ep = plan_expert(min(p.cumsums[e + 1], p.msum) - min(p.cumsums[e], p.msum), pl.kc);
    const int ne = tpe * ep.splits;
    bc += (int64_t)ne * item_cost<THREADS>(ep.chunk);
    bn += ne;
    if (ep.splits > 1) bs += ne, bt += tpe;
  }
  if (threadIdx.x == THREADS - 1)
    pl.cost[p.N] = bc, pl.items[p.N] = bn, pl.slots[p.N] = bs, pl.ctiles[p.N] = bt;
  __syncthreads();
  return pl;
}

// The same when no expert is cut: only the cost prefix sums are needed, an expert's items
// are its tpe tiles.
template <int THREADS>
__device__ __forceinline__ Plan build_cost_plan(const WgradArgs& p, int tpe) {
  Plan pl;
  pl.cost = (int64_t*)dyn_lds();
  pl.items = pl.slots = pl.ctiles = nullptr;
  pl.kc = 0x7fffffff;
  int64_t* wave_tot = pl.cost + p.N + 1;
  const int per = (p.N + THREADS - 1) / THREADS;  // experts per thread, contiguous
  const int e0 = min((int)threadIdx.x * per, p.N), e1 = min(e0 + per, p.N);
  auto cost_of = [&](int e) {
    const int rows = min(p.cumsums[e + 1], p.msum) - min(p.cumsums[e], p.msum);
    return (int64_t)tpe * item_cost<THREADS>((rows + kBK - 1) / kBK);
  };
  int64_t mine = 0;
  for (int e = e0; e < e1; ++e) mine += cost_of(e);
  int64_t incl = mine;  // inclusive scan over the wave, then over the waves
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t v = __shfl_up(incl, o);
    if ((int)(threadIdx.x & 63) >= o) incl += v;
  }
  if ((threadIdx.x & 63) == 63) wave_tot[threadIdx.x >> 6] = incl;
  __syncthreads();
  int64_t run = incl - mine;
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) run += wave_tot[w];
  for (int e = e0; e < e1; ++e) {
    pl.cost[e] = run;
    run += cost_of(e);
  }
  if (threadIdx.x == THREADS - 1) pl.cost[p.N] = run;
  __syncthreads();
  return pl;
}

// values read back from LDS are the same in every lane; tell the compiler so
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// A routing with more pairs than sorted rows (cumsums[N] > Msum) got an empty tile table: the
// GEMMs before this one wrote nothing, so no expert has rows to contract over and every weight
// gradient is zero.  Row counts are clamped to p.msum everywhere: clamp them to nothing.
__device__ __forceinline__ void drop_rows_of_an_overflowed_routing(WgradArgs& p) {
  if (load_uniform(p.cumsums + p.N) > p.msum) p.msum = 0;
}

// Persistent workgroups.  id%8 is the XCD a workgroup lands on.  Work items are numbered
// expert by expert and cut into 8 contiguous runs of equal estimated cost (an item costs its
// k-stages plus the epilogue), one per XCD, whose workgroups walk the run with a stride: an
// expert's rows are then fetched from HBM by one L2 (two for an expert that straddles a cut)
// and re-read from there by all of its tiles.  An expert with many times the rows of the
// others would make single tiles as long as a workgroup's whole share, so its rows are cut
// into pieces; the pieces of a tile go to the workspace in fp32 and wgrad_reduce_kernel adds
// them up.
// CUT = false is the launch in which no expert can reach the cutting length (the host knows:
// an expert holds at most M rows): the bookkeeping of pieces is compiled out.
template <bool CUT, int THREADS>
struct WorkItems {
  const WgradArgs& p;
  int tpe, stride, kc, g_end, pos;
  int ex = 0, ex_first = 0, ex_slot = 0;  // the expert that holds item `pos`; later ones are reached by walking forward
  int ex_rb = 0, ex_re = 0, ahead = 0;
  ExpertPlan ep = {0, 1, 0};
  __device__ __forceinline__ explicit WorkItems(const WgradArgs& p_) : p(p_), tpe(p_.tiles_x * p_.tiles_y), stride(gridDim.x >> 3) {
    const int xcd = blockIdx.x & 7;
    const Plan pl = CUT ? build_plan<THREADS>(p, tpe) : build_cost_plan<THREADS>(p, tpe);
    if constexpr (THREADS == kSpanThreads) find_empty(pl);
    kc = CUT ? uniform(pl.kc) : 0x7fffffff;
    auto items_before = [&](int e) { return CUT ? pl.items[e] : e * tpe; };

    // first item whose cost interval starts at or after `c`
    auto item_at = [&](int64_t c) -> int {
      if (c >= pl.cost[p.N]) return items_before(p.N);
      int lo = 0, hi = p.N;  // cost[lo] <= c < cost[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pl.cost[mid] <= c) lo = mid; else hi = mid;
      }
      const int64_t each = (pl.cost[lo + 1] - pl.cost[lo]) / (items_before(lo + 1) - items_before(lo));
      return items_before(lo) + (int)((c - pl.cost[lo] + each - 1) / each);
    };
    const int64_t total_cost = pl.cost[p.N];
    const int total = items_before(p.N), all = gridDim.x;
    int2 run;
    if (total <= all)  // one each
      run = {total * xcd / 8, total * (xcd + 1) / 8};
    else if (THREADS != kSpanThreads || !whole_rounds(pl, items_before, run))
      run = {item_at(total_cost * xcd / 8), item_at(total_cost * (xcd + 1) / 8)};
    g_end = uniform(run.y);
    pos = uniform(run.x) + (int)(blockIdx.x >> 3);
    if constexpr (CUT) {
      int lo = 0, hi = p.N;  // items[lo] <= pos < items[hi] (if pos is an item at all)
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pl.items[mid] <= pos) lo = mid; else hi = mid;
      }
      ex = uniform(lo);
      ex_first = uniform(pl.items[ex]);  // first item of expert ex
      ex_slot = uniform(pl.slots[ex]);   // first partial tile of expert ex
    }
    __syncthreads();  // the rings are handed to the transfers
    if constexpr (CUT) {
      ex_rb = min(load_uniform(p.cumsums + ex), p.msum);
      ex_re = min(load_uniform(p.cumsums + ex + 1), p.msum);
      ep = plan_expert(ex_re - ex_rb, kc);
      // end of the next expert's rows, requested one expert ahead so that moving on does not wait
      ahead = load_uniform(p.cumsums + min(ex + 2, p.N));
    }
  }
  bool some_empty = false;  // experts
  __device__ __forceinline__ void find_empty(const Plan& pl) {
    for (int e0 = 0; e0 < p.N; e0 += 64) {
      const int e = min(e0 + lane_id(), p.N - 1);
      some_empty = some_empty || __ballot(pl.cost[e + 1] == pl.cost[e]) != 0;
    }
  }
  // Where a workgroup has few items, runs of equal cost leave rounds of the XCD's workgroups nearly empty: a run
  // of 99 tiles of 16384 rows takes four rounds, not three.  Instead each XCD takes as many rounds as fit a time
  // limit, and the limit is the least of 64, one tried by each lane, with which the items end in the last XCD.
  // 16384 tokens, 64 experts of which ten hold nearly all rows, D = 2048, H = 1408: from 75 to 94 % of the
  // workgroups' time used.
  template <class Before>
  __device__ __forceinline__ bool whole_rounds(const Plan& pl, Before items_before, int2& run) const {
    constexpr int kFewRounds = 8, kShareOfWalk = 8;  // the walk takes 0.1 us per expert, a unit of cost 0.8 us
    const int lane = lane_id(), xcd = blockIdx.x & 7;
    const int64_t share = pl.cost[p.N] / (8 * stride);
    if (share < (int64_t)kShareOfWalk * p.N || (stride & (stride - 1)) != 0) return false;
    auto items_of = [&](int e) { return e < p.N ? items_before(e + 1) - items_before(e) : 0; };
    auto each = [&](int e) {
      return e < p.N ? (int)((float)(pl.cost[e + 1] - pl.cost[e]) / (float)items_of(e) + 0.5f) : 1;
    };
    int most = 0;
    for (int e = lane; e < p.N; e += 64) most = max(most, each(e));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
    if ((int64_t)kFewRounds * most <= share) return false;
    const int limit = (int)(share + share * lane / 64);
    const int total = items_before(p.N), per_round = __builtin_ctz(stride);
    int x = 0, load = 0, left = 0;  // of the run of XCD x: cost of its rounds, items left of the last one
    int open = 0;                   // cost of that one
    int first = 0;                  // next item
    run = {xcd == 0 ? 0 : total, total};
    for (int e0 = 0; e0 < p.N; e0 += 64) {
      const int my_items = items_of(e0 + lane), my_cost = each(e0 + lane);
      for (int i = 0; i < min(64, p.N - e0); ++i) {
        int n = __builtin_amdgcn_readlane(my_items, i);
        const int c = __builtin_amdgcn_readlane(my_cost, i);
        const float inv = 1.0f / (float)max(c, 1);
        if (left > 0) load += max(0, c - open), open = max(open, c);
        else open = c;
        while (n > 0 && x < 8) {
          // items without rows take their places in the rounds, but no time
          const int room = left + ((c > 0 ? (int)min((float)max(0, limit - load) * inv, 1e7f) : 10000000) << per_round);
          if (n <= room) {
            const int rounds = (max(0, n - left) + stride - 1) >> per_round;
            if (rounds > 0) open = c;
            load += rounds * c;
            left += (rounds << per_round) - n;
            first += n, n = 0;
          } else {
            first += room, n -= room, ++x;
            if (x == xcd) run.x = first;
            if (x == xcd + 1) run.y = first;
            load = left = 0;
            open = c;
          }
        }
      }
    }
    const uint64_t fits = __ballot(x < 8);
    if (fits == 0) return false;
    const int best = __builtin_ctzll(fits);
    run = {__shfl(run.x, best), __shfl(run.y, best)};
    return true;
  }
  __device__ __forceinline__ WTile next() {
    WTile t = {};
    t.valid = pos < g_end;
    if (!t.valid) return t;
    if constexpr (!CUT) {
      const int expert = pos / tpe;
      t.q = pos - expert * tpe;
      pos += stride;
      t.expert = expert;
      t.rows.rb = min(load_uniform(p.cumsums + expert), p.msum);
      t.rows.re = min(load_uniform(p.cumsums + expert + 1), p.msum);
      t.rows.prow = padded_start(t.rows.rb, expert);
      t.slot = -1;
      return t;
    }
    while (pos >= ex_first + tpe * ep.splits && ex + 1 < p.N) {
      ex_first += tpe * ep.splits;
      if (ep.splits > 1) ex_slot += tpe * ep.splits;
      ++ex;
      ex_rb = ex_re;
      ex_re = min(ahead, p.msum);
      ahead = load_uniform(p.cumsums + min(ex + 2, p.N));
      ep = plan_expert(ex_re - ex_rb, kc);
    }
    const int it = pos - ex_first, piece = it / tpe;
    pos += stride;
    t.expert = ex;
    t.q = it - piece * tpe;
    t.rows.rb = min(ex_re, ex_rb + piece * ep.chunk * kBK);
    t.rows.re = min(ex_re, t.rows.rb + ep.chunk * kBK);
    t.rows.prow = padded_start(ex_rb, ex) + (t.rows.rb - ex_rb);
    t.slot = ep.splits > 1 ? ex_slot + it : -1;
    return t;
  }
};

// ---- 32 rows a stage, 8 wavefronts (gemm_tile.hpp): few rows per expert ------------------------------
// Per wave and k-step the 4-fragment side of the 128 x 64 wave tile reads twice the LDS bytes of
// the 2-fragment side, so the transposed operand is given the 4 fragments: it is the M side
// (FM=4, FN=2) when A is transposed and the N side (FM=2, FN=4) when B is.
namespace tile {

constexpr int kStages = 4;  // ring depth
constexpr int kRingBytes = kStages * 2 * TLayout::LDS_ELEMS * 2;  // every operand kind: 16 KiB per stage
constexpr size_t kWgradLds = kRingBytes + kEpilogueLds;  // stage ring + per-wave store staging
static_assert((size_t)(kMaxWgradExperts + 1) * 20 + 512 <= kRingBytes, "prefix sums overlay the ring");

// "rows" operand of a work item: the gathered / sorted rows [rb, re)
struct RowsOperand : TGatherDmaT<true, kStages - 1> {
  __device__ __forceinline__ void begin_piece(const int32_t* gather_, int64_t ld_, int rb, int re, int) {
    set_rows(gather_, ld_, rb, re);
  }
};
// "k-blocked" operand: sorted rows (no gather) of a matrix stored in blocks of 32 features,
// feature f of row r at mat[((f / 32) * ld + r) * 32 + f % 32], ld = rows of the matrix (gz, as
// the SwiGLU backward writes it for dL/dx).  Rows are the contraction index, as in the row layout,
// and go through the same transposing LDS reads; the 32 rows x 32 features of a block are 2 KiB
// of consecutive memory.
struct BlockedRowsOperand : TGatherDmaT<false, kStages - 1> {
  int64_t nrows;
  __device__ __forceinline__ void begin_piece(const int32_t*, int64_t ld_, int rb, int re, int) {
    nrows = ld_;
    set_rows(nullptr, 32, rb, re);  // row pitch: 32 elements
  }
  // features [col0, col0+256) (col0 a multiple of 256); features >= ncols are clamped to col0
  __device__ __forceinline__ void set_cols(const bf16* mat_, int col0, int ncols) {
    mat = mat_ + ((int64_t)(col0 >> 5) * nrows + row_begin) * 32;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      int krow, c;
      L::lane_piece(j, krow, c);
      const int cc = col0 + c < ncols ? c : 0;
      colb[j] = (uint32_t)(((int64_t)(cc >> 5) * nrows * 32 + (cc & 31)) * 2);
    }
  }
};

// "transposed" operand: groups of 32 padded sorted rows, feature-major inside a group: feature f
// of padded sorted row p at mat[(p / 32) * ld * 32 + f * 32 + p % 32], ld >= number of features.
// The 256 features x 32 rows of one stage are 16 KiB of consecutive memory.
struct TransposedOperand {
  using R = RDma<256>;
  static constexpr int NCH = R::NCH;
  static constexpr int LDS_ELEMS = R::LDS_ELEMS;
  static_assert(LDS_ELEMS == TLayout::LDS_ELEMS, "same stage size as the other operand kind");
  R r;
  int64_t gstride;  // elements between consecutive 32-row groups
  int g0;           // group of the first row of the piece
  __device__ __forceinline__ void begin_piece(const int32_t*, int64_t ld_, int, int, int prow) {
    gstride = ld_ * 32;
    g0 = prow >> 5;
  }
  // features [f0, f0+256) of the matrix; features >= nfeat are clamped to the last one
  __device__ __forceinline__ void set_cols(const bf16* mat, int f0, int nfeat) {
    r.init(mat + (int64_t)g0 * gstride + (int64_t)f0 * 32,
           [&](int row, int) { return (uint32_t)min(row, nfeat - 1 - f0) * 64u; });
  }
  __device__ __forceinline__ void issue(int kt, uint32_t stage) {
    const int w = wave_id();
    const bf16* b = r.base + (int64_t)kt * gstride;
#pragma unroll
    for (int j = 0; j < NCH; ++j) dma16(b, r.off[j], stage + (j * kWaves + w) * (kChunkElems * 2));
  }
  template <int S>
  __device__ __forceinline__ void issue_head(uint32_t stage) { issue(S, stage); }
  static __device__ __forceinline__ bf16x8 frag(const bf16* stage, int c0, int kk) { return R::frag(stage, c0, kk); }
};

// How the 8 waves share the 256 x 256 output tile: FM x FN fragments of 32 x 32 per wave.
template <int FM, int FN>
struct WaveTile {
  static_assert(FM * FN == 8 && (FM == 4 || FM == 2), "128 x 64 or 64 x 128 per wave");
  static constexpr int WAVES_N = 256 / (32 * FN);  // waves side by side
  int m_org[FM], n_org[FN];
  __device__ __forceinline__ WaveTile() {
    const int wave = wave_id(), wm = wave / WAVES_N, wn = wave % WAVES_N;
#pragma unroll
    for (int i = 0; i < FM; ++i) m_org[i] = wm * (32 * FM) + 32 * i;
#pragma unroll
    for (int j = 0; j < FN; ++j) n_org[j] = wn * (32 * FN) + 32 * j;
  }
};

// bf16 store of one output tile from the accumulators (non-temporal: a weight gradient is
// not read again by this kernel); two fragments (64 columns) go through the staging area at a time
template <int FM, int FN>
__device__ __forceinline__ void store_gw_tile(const WgradArgs& p, RowStager<2>& stager,
                                              f32x16 (&acc)[FN][FM], int expert, int x0, int y0t,
                                              const WaveTile<FM, FN>& wt) {
  bf16* out = p.gw + (int64_t)expert * p.X * p.Y;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int f0 = 0; f0 < FN; f0 += 2) {
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          stager.put(f, qd, pack_bf16x4(acc[f0 + f][i][4 * qd], acc[f0 + f][i][4 * qd + 1],
                                        acc[f0 + f][i][4 * qd + 2], acc[f0 + f][i][4 * qd + 3]));
      const int y0 = y0t + wt.n_org[f0];  // first output column of these two fragments
      stager.flush<true>([&](int row, int col) -> bf16* {
        const int x = x0 + wt.m_org[i] + row;
        if (x >= p.X || y0 + col >= p.Y) return nullptr;
        return out + (int64_t)x * p.Y + y0 + col;
      });
    }
  }
}

// A partial tile is kept in accumulator order: per wave, per fragment, 4 x (64 lanes x 16 B).
template <int FM, int FN>
__device__ __forceinline__ f32x4* partial_piece(float* ws, int slot, int i, int f, int qd) {
  const int wave = wave_id(), lane = threadIdx.x & 63;
  return (f32x4*)(ws + (int64_t)slot * (BX * BY)) +
         ((((wave * FM + i) * FN + f) * 4 + qd) * 64 + lane);
}

template <bool CUT, class AOp, class BOp, int FM, int FN>
__device__ __forceinline__ void wgrad_tiles(WgradArgs p) {
  drop_rows_of_an_overflowed_routing(p);
  using Ring = StageRing<AOp, BOp, kStages>;
  static_assert(Ring::BYTES == kRingBytes, "ring size assumed by the launch");
  const ClockTrace trace(p.clk);
  Ring ring(dyn_lds());
  WorkItems<CUT, kThreads> items(p);
  // With values from the start: where members had none, the compiler kept the ids that RowsOperand asks for a stage
  // ahead in vector registers, and moving them there waits for their loads at once (Wl1 gradient of 10880 rows in 32
  // experts, load falling as rank^-0.5, D = 1024, H = 512: 51 us where 41 are due).
  AOp A = {};
  BOp B = {};
  int cur_rb = -1, cur_re = -1;
  // the rows of a piece (and the ids of the first of them) are looked up when the workgroup
  // moves on to a new piece; every tile of the piece then reuses them
  auto start = [&](const WTile& t) {
    if (t.rows.re <= t.rows.rb) return;  // no rows: nothing to load, zeros are stored
    if (t.rows.rb != cur_rb || t.rows.re != cur_re) {
      cur_rb = t.rows.rb;
      cur_re = t.rows.re;
      A.begin_piece(p.ga, p.lda, t.rows.rb, t.rows.re, t.rows.prow);
      B.begin_piece(p.gb, p.ldb, t.rows.rb, t.rows.re, t.rows.prow);
    }
    A.set_cols(p.a, t.x0, p.X);
    B.set_cols(p.b, t.y0, p.Y);
    gemm_issue_first(A, B, ring, (t.rows.re - t.rows.rb + kBK - 1) / kBK);
  };
  const WaveTile<FM, FN> wt;
  RowStager<2> stager(dyn_lds() + kStages * Ring::STAGE);

  auto next_tile = [&] {
    WTile t = items.next();
    t.x0 = uniform(t.q / p.tiles_y * BX);
    t.y0 = uniform(t.q % p.tiles_y * BY);
    t.rows = {uniform(t.rows.rb), uniform(t.rows.re), uniform(t.rows.prow)};
    return t;
  };
  WTile tc = next_tile();
  if (!tc.valid) {
    trace.finish();
    return;
  }
  start(tc);
  while (true) {
    f32x16 acc[FN][FM];
    zero_acc<FM, FN>(acc);
    const int ktiles = (tc.rows.re - tc.rows.rb + kBK - 1) / kBK;
    const int ktail = tc.rows.re - tc.rows.rb - (ktiles - 1) * kBK;
    const WTile nx = next_tile();
    if (ktiles > 0)
      gemm_mainloop<AOp, BOp, kStages, FM, FN, FM>(A, B, acc, ktiles, ring, wt.m_org, wt.n_org, [] {}, ktail);
    if (nx.valid) start(nx);

    if (!CUT || tc.slot < 0) {
      store_gw_tile<FM, FN>(p, stager, acc, tc.expert, tc.x0, tc.y0, wt);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int f = 0; f < FN; ++f)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            f32x4 v = {acc[f][i][4 * qd], acc[f][i][4 * qd + 1], acc[f][i][4 * qd + 2],
                       acc[f][i][4 * qd + 3]};
            *partial_piece<FM, FN>(p.ws, tc.slot, i, f, qd) = v;
          }
    }
    if (!nx.valid) break;
    tc = nx;
  }
  trace.finish();
}

template <bool CUT, class AOp, class BOp, int FM, int FN>
__global__ __launch_bounds__(kThreads, 2) void wgrad_kernel(WgradArgs p) {
  wgrad_tiles<CUT, AOp, BOp, FM, FN>(p);
}

// The end of a small call's backward, three products that do not need each other and dL/ds, in one launch: the workgroups of a
// part start on the CUs that the part before it leaves, where a launch would wait for its last tile and then find its work.
// The Wl1 gradient first, the longest; then dL/dx, whose few long tiles would end the launch late, or behind both weight gradients
// where the weights, or their gradients, do not fit the last-level cache (kBeyondCache): between them it took even loads
// past the time of four launches.  A step in us, four launches | dL/dx second | last: 1024 tokens, D = 1024, H = 512, N = 32, K = 4
// 153 | 142 | 142; 307, 512, 1728, 32, 6 186 | 163 | 170; 868, 256, 1152, 128, 6, two of them shared, 320 | 271 | 280; 128, 128, 64, 8,
// 2, bound by the host's launches, 117 | 108 | 108; past the line 1500, 2048, 512, 96, 4 517 | 529 | 515; 64, 4096, 1408, 128, 8
// 2715 | 2754 | 2682; 1024, 1024, 512, 128, 8 347 | 352 | 341; 195, 1792, 2016, 64, 6 949 | 962 | 924; and, loads that fall as
// rank^-1.8, 700, 2048, 768, 128, 8 677 | 668 | 641; 1500, 2048, 512, 96, 4 417 | 372 | 377; 3000, 2048, 1408, 128, 1 716 | 634 | 666.
constexpr unsigned kTailParts = 4;
struct TailArgs {
  WgradArgs w1, w2;
  DxArgs dx;
  GsTokensArgs gs;  // gs.gs == nullptr: not wanted
  unsigned dx_part;
};
__global__ __launch_bounds__(kThreads, 2) void backward_tail_kernel(TailArgs p) {
  if (blockIdx.y == 0) {
    wgrad_tiles<false, RowsOperand, BlockedRowsOperand, 4, 2>(p.w1);
  } else if (blockIdx.y == p.dx_part) {
    dgrad_x_short(p.dx);
  } else if (blockIdx.y < kTailParts - 1) {
    wgrad_tiles<false, TransposedOperand, RowsOperand, 4, 2>(p.w2);
  } else if (p.gs.gs != nullptr) {
    static_assert(kGsThreads == kThreads, "the same workgroups");
    const int across = (p.gs.M + kGsTileTokens - 1) / kGsTileTokens, tiles = across * ((p.gs.N + kGsTileExperts - 1) / kGsTileExperts);
    for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
      gs_scatter_tokens(p.gs, t % across, t / across, *(GsTile*)dyn_lds());
      __syncthreads();
    }
  }
}

// Adds up the partial tiles of the experts that wgrad_kernel cut into pieces and stores the
// bf16 result; one workgroup per output tile, same register layout as the GEMM.
template <int FM, int FN>
__global__ __launch_bounds__(kThreads) void wgrad_reduce_kernel(WgradArgs p) {
  drop_rows_of_an_overflowed_routing(p);
  const int tpe = p.tiles_x * p.tiles_y;
  const Plan pl = build_plan<kThreads>(p, tpe);
  const int ncut = pl.ctiles[p.N];
  const WaveTile<FM, FN> wt;
  RowStager<2> stager((bf16*)((char*)dyn_lds() + kRingBytes));
  for (int t = blockIdx.x; t < ncut; t += gridDim.x) {
    int lo = 0, hi = p.N;  // ctiles[lo] <= t < ctiles[hi]; the last such lo is the cut expert
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (pl.ctiles[mid] <= t) lo = mid; else hi = mid;
    }
    const int q = t - pl.ctiles[lo];
    const int splits = (pl.slots[lo + 1] - pl.slots[lo]) / tpe;
    f32x16 acc[FN][FM];
    zero_acc<FM, FN>(acc);
    for (int piece = 0; piece < splits; ++piece) {
      const int slot = pl.slots[lo] + piece * tpe + q;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int f = 0; f < FN; ++f)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const f32x4 v = *partial_piece<FM, FN>(p.ws, slot, i, f, qd);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[f][i][4 * qd + r] += v[r];
          }
    }
    store_gw_tile<FM, FN>(p, stager, acc, lo, (q / p.tiles_y) * BX, (q % p.tiles_y) * BY, wt);
  }
}

template <class AOp, class BOp, int FM, int FN>
int launch(const WgradArgs& a, bool can_cut, hipStream_t st) {
  const int grid = persistent_grid();
  static LdsLimit once, once_cut, once_reduce;
  if (!can_cut) {
    if (!allow_lds(wgrad_kernel<false, AOp, BOp, FM, FN>, kWgradLds, once)) return MOMOE_ERR_LAUNCH;
    wgrad_kernel<false, AOp, BOp, FM, FN><<<grid, kThreads, kWgradLds, st>>>(a);
  } else {
    if (!allow_lds(wgrad_kernel<true, AOp, BOp, FM, FN>, kWgradLds, once_cut) ||
        !allow_lds(wgrad_reduce_kernel<FM, FN>, kWgradLds, once_reduce))
      return MOMOE_ERR_LAUNCH;
    wgrad_kernel<true, AOp, BOp, FM, FN><<<grid, kThreads, kWgradLds, st>>>(a);
    wgrad_reduce_kernel<FM, FN><<<grid, kThreads, kWgradLds, st>>>(a);
  }
  return launch_status();
}

}  // namespace tile

// ---- 64 rows a stage, 4 wavefronts (gemm_span.hpp) --------------------------------------------------------
// With 512 rows per expert a tile is 8 stages and then 128 KiB to store, so most of what a drain at each
// tile would cost is in these launches.
namespace span {

// LDS that the prefix sums may take; behind it the reduction's staging
constexpr int kPlanLds = kSpanLds - kSpanWaves * kStagingElems * sizeof(bf16);
static_assert((size_t)(kMaxWgradExperts + 1) * 20 + 512 <= kPlanLds, "prefix sums overlay the rings");

// Common to the operands: set_tile() says where a tile's stages come from; request() starts the loads
// that the deposits of a stage need, a stage ahead, those of the span given to restart() in turn; begin(span, t)
// precedes the deposits of stage t, prepare<j>() uses up what was loaded for one, deposit<j>(slot) requests it.  Rows past the end are the
// expert's last one: the M side's zeros meet finite numbers if the expert's are finite.  The stages of a
// span without rows take row and token 0: the list may hold nothing yet.

// "rows" operand.  LDS [64][256] as SpanCols; wave w deposits k-rows [16 w, 16 w + 16), two a time.  The
// ids of gathered rows are wave-uniform and come through scalar loads, 16 at once while all exist.
// Sources are a wave-uniform base plus a 32-bit byte offset per lane: the matrix for a gathered
// operand, the span's first row otherwise, so (number of tokens) x (row pitch) must stay below 4 GiB.
struct RowsOperand {
  using L = SpanCols<>;
  using Lane = L::Lane;
  static constexpr int DEP = L::DEP, ELEMS = L::ELEMS, ROWS = 2 * DEP;
  typedef int32_t ids_t __attribute__((ext_vector_type(ROWS), aligned(4)));
  const bf16* mat;
  uint32_t ldb;  // bytes between rows
  const int32_t* gather;
  uint32_t colb[4];  // byte offset of this lane's columns, by the swizzle of its k-row
  ids_t next;        // of the stage whose deposits come next: tokens, or rows from the span's first one
  uint32_t off[DEP]; // byte offsets of its prepared deposits
  int at, origin, last, some;  // row of this wave's next id, the span's first and last, all ones if it has any
  uint32_t upper;    // all ones in the lanes that fetch the second k-row of a deposit
  static __device__ __forceinline__ int wave_offset() { return wave_id() * (ROWS * 512); }
  __device__ __forceinline__ RowsOperand(const bf16* mat_, int64_t ld, const int32_t* gather_)
      : mat(mat_), ldb((uint32_t)(ld * 2)), gather(gather_), upper(lane_id() >= 32 ? 0xFFFFFFFFu : 0u) {}
  // the requests that follow are for the span's stages in turn
  __device__ __forceinline__ void restart(const Span& sp) {
    at = sp.rb + wave_id() * ROWS;
    origin = sp.rb;
    last = max(sp.re - 1, 0);
    some = sp.re > 0 ? -1 : 0;
  }
  __device__ __forceinline__ void request() {
    if (gather == nullptr) {  // kernel-uniform
#pragma unroll
      for (int i = 0; i < ROWS; ++i) next[i] = min(at + i, last) - origin;
    } else if (at + ROWS - 1 <= last) {
      next = *(const ids_t __attribute__((address_space(4)))*)(gather + at);
    } else {
#pragma unroll
      for (int i = 0; i < ROWS; ++i) next[i] = load_uniform(gather + min(at + i, last));
#pragma unroll
      for (int i = 0; i < ROWS; ++i) next[i] &= some;
    }
    at += kSpan;
  }
  // columns [col0, col0 + 256) of the matrix; columns >= ncols are clamped to column 0
  __device__ __forceinline__ void set_tile(const bf16* mat_, const Span& sp, int col0, int ncols) {
    mat = gather ? mat_ : (const bf16*)((const char*)mat_ + (int64_t)sp.rb * ldb);
    const int l = fresh_lane();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int krow = 2 * (q & 1) + 8 * (q >> 1) + (l >> 5);  // (its wave's first k-row does not matter)
      const int c = col0 + ((l & 31) ^ L::swz(krow)) * 8;
      colb[q] = (uint32_t)(c < ncols ? c : 0) * 2;
    }
  }
  __device__ __forceinline__ void begin(const Span&, int) {}
  template <int j>
  __device__ __forceinline__ void prepare() {
    const uint32_t lo = (uint32_t)next[2 * j] * ldb, hi = (uint32_t)next[2 * j + 1] * ldb;
    off[j] = lo + (upper & (hi - lo)) + colb[(j & 1) + 2 * (j >> 2)];
    settle(off[j]);  // (here, between products, and not where it is used)
  }
  template <int j>
  __device__ __forceinline__ void deposit(uint32_t slot) const {
    dma16_at<j * 1024>(mat, off[j], slot);
  }
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) { return L::frag(slot, ln, i, h); }
};

// "k-blocked" operand: sorted rows (no gather) of a matrix stored in blocks of 32 features,
// feature f of row r at mat[((f / 32) * ld + r) * 32 + f % 32], ld = rows of the matrix (gz, as
// the SwiGLU backward writes it for dL/dx).  LDS as above; a deposit is k-rows 8 j + 2 w and the next.
struct BlockedRowsOperand {
  using L = SpanCols<>;
  using Lane = L::Lane;
  static constexpr int DEP = L::DEP, ELEMS = L::ELEMS;
  const bf16 *mat, *src;
  int64_t nrows;
  uint32_t colb[2];
  int last;  // of the rows of the stage at hand
  static __device__ __forceinline__ int wave_offset() { return wave_id() * 1024; }
  __device__ __forceinline__ BlockedRowsOperand(const bf16* mat_, int64_t ld, const int32_t*) : mat(mat_), nrows(ld) {}
  __device__ __forceinline__ void restart(const Span&) {}
  __device__ __forceinline__ void request() {}
  // features [col0, col0+256) (col0 a multiple of 256); features >= ncols are clamped to col0
  __device__ __forceinline__ void set_tile(const bf16* mat_, const Span&, int col0, int ncols) {
    mat = mat_ + (int64_t)(col0 >> 5) * nrows * 32;
    const int l = fresh_lane();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int krow = 8 * q + 2 * wave_id() + (l >> 5);
      const int c = ((l & 31) ^ L::swz(krow)) * 8, cc = col0 + c < ncols ? c : 0;
      colb[q] = (uint32_t)(((int64_t)(cc >> 5) * nrows * 32 + (cc & 31)) * 2);
    }
  }
  template <int j>
  __device__ __forceinline__ void prepare() {}
  __device__ __forceinline__ void begin(const Span& sp, int t) {
    const int first = min(sp.rb + t * kSpan, max(sp.re - 1, 0));
    src = mat + (int64_t)first * 32;
    last = max(sp.re - 1, 0) - first;
  }
  template <int j>
  __device__ __forceinline__ void deposit(uint32_t slot) const {
    const int krow = min(8 * j + 2 * wave_id() + (lane_id() >> 5), last);
    dma16_at<L::STEP * 512 * j>(src, colb[j & 1] + (uint32_t)krow * 64, slot);
  }
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) { return L::frag(slot, ln, i, h); }
};

// "transposed" operand: groups of 32 padded sorted rows, feature-major inside a group: feature f
// of padded sorted row p at mat[(p / 32) * ld * 32 + f * 32 + p % 32], ld >= number of features.
// LDS as SpanBlockedRows<256>.
struct TransposedOperand {
  using L = SpanBlockedRows<256>;
  using Lane = L::Lane;
  static constexpr int DEP = L::DEP, ELEMS = L::ELEMS;
  const bf16 *mat, *src;
  int64_t gstride, second;  // elements between groups, to the stage's second one
  uint32_t off[L::PER_HALF];
  static __device__ __forceinline__ int wave_offset() { return wave_id() * 1024; }
  __device__ __forceinline__ TransposedOperand(const bf16* mat_, int64_t ld, const int32_t*) : mat(mat_), gstride(ld * 32) {}
  __device__ __forceinline__ void restart(const Span&) {}
  __device__ __forceinline__ void request() {}
  // features [f0, f0+256) of the matrix; features >= nfeat are clamped to the last one
  __device__ __forceinline__ void set_tile(const bf16* mat_, const Span&, int f0, int nfeat) {
    mat = mat_ + (int64_t)f0 * 32;
    const int l = fresh_lane();
#pragma unroll
    for (int q = 0; q < L::PER_HALF; ++q) {
      const int row = (q * kSpanWaves + wave_id()) * 16 + (l >> 2);
      off[q] = (uint32_t)min(row, nfeat - 1 - f0) * 64 + (((l & 3) ^ L::swz(row)) * 16);
    }
  }
  template <int j>
  __device__ __forceinline__ void prepare() {}
  __device__ __forceinline__ void begin(const Span& sp, int t) {
    const int groups = (sp.re - sp.rb + 31) >> 5, g = max(0, min(2 * t, groups - 1));
    src = mat + (int64_t)((sp.prow >> 5) + (groups > 0 ? g : 0)) * (groups > 0 ? gstride : 0);
    second = g + 1 < groups ? gstride : 0;
  }
  template <int j>
  __device__ __forceinline__ void deposit(uint32_t slot) const {
    constexpr int h = j / L::PER_HALF, q = j % L::PER_HALF;
    dma16_at<h * (256 * kHalf * 2) + q * kSpanWaves * 1024>(h ? src + second : src, off[q], slot);
  }
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) { return L::frag(slot, ln, i, h); }
};

constexpr int FM = WideSpan::FM, FN = WideSpan::FN;  // a wave holds 128 x 128 of the tile, waves 2 x 2
typedef f32x4 TileAcc[FN][FM];
__device__ __forceinline__ int wave_row() { return wave_id() / 2 * 128; }
__device__ __forceinline__ int wave_col() { return wave_id() % 2 * 128; }

// The q-th output tile of an expert: in bands of four, each band crossing all columns.  The 32 workgroups of
// an XCD then share four blocks of A and eight of B.
__device__ __forceinline__ void place_tile(const WgradArgs& p, WTile& t) {
  const int q = t.q, band = q / (kBandTiles * p.tiles_y), in = q - band * (kBandTiles * p.tiles_y);
  const int high = min(kBandTiles, p.tiles_x - band * kBandTiles);
  t.x0 = (band * kBandTiles + in % high) * BX;
  t.y0 = in / high * BY;
}

// bf16 store of one output tile (non-temporal: a weight gradient is not read again by this kernel)
__device__ __forceinline__ void store_gw_tile(const WgradArgs& p, TileAcc& acc, int expert, int x0, int y0, bf16* staging) {
  const int x = x0 + wave_row();
  store_rows<true>(acc, staging, p.gw + (int64_t)expert * p.X * p.Y, x, p.X - x, p.Y, y0 + wave_col(), fresh_lane(),
                   [](int) { return 1.0f; });
}

// Zeros in one output tile
__device__ __forceinline__ void zero_gw_tile(const WgradArgs& p, const WTile& t) {
  const int l = fresh_lane(), row = 2 * wave_id() + (l >> 5), col = (l & 31) * 8;
  bf16* const first = p.gw + ((int64_t)t.expert * p.X + t.x0) * p.Y + t.y0;  // uniform
  const bf16x8 zero = {};
#pragma unroll 4
  for (int r = 0; r < BX; r += 2 * kSpanWaves)
    store16<true>(first + (int64_t)r * p.Y, ((uint32_t)row * (uint32_t)p.Y + col) * 2, t.x0 + r + row < p.X && t.y0 + col < p.Y, zero);
}

// A partial tile is kept in accumulator order: per wave, per accumulator, 64 lanes x 16 B.
__device__ __forceinline__ f32x4* partial_piece(float* ws, int slot, int f, int i) {
  return (f32x4*)(ws + (int64_t)slot * (BX * BY)) + ((wave_id() * FN + f) * FM + i) * 64;
}

// Stored from the accumulation registers they are in: copies to vector registers, shared with the tile's other
// store, had 84 of them spilled.  (The compiler does not know that a piece of assembly reads products:
// 32 cycles cover those in flight.)
__device__ __forceinline__ void store_partial(const WgradArgs& p, TileAcc& acc, int slot) {
  const uint32_t lane = fresh_lane() * 16;
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int f = 0; f < FN; ++f)
#pragma unroll
    for (int i = 0; i < FM; ++i)
      asm volatile("global_store_dwordx4 %0, %1, %2" ::"v"(lane), "a"(acc[f][i]), "s"(partial_piece(p.ws, slot, f, i)) : "memory");
}

// A in a ring of two stages, B in one of three (gemm_span.hpp).
template <bool CUT, class AOp, class BOp>
__global__ __launch_bounds__(kSpanThreads, 1) void wgrad_kernel(WgradArgs p) {
  drop_rows_of_an_overflowed_routing(p);
  const ClockTrace trace(p.clk);
  WorkItems<CUT, kSpanThreads> items(p);
  // Tiles of experts without rows: stores that nothing waits for, behind the loop, dealt out to all workgroups.  As two
  // stages of the loop such a tile waited for the stores of the tile before it, for the stages' transfers and for its
  // own stores; left in the runs of the XCDs, behind the loop, they were stored at the rate of the one or two XCDs that
  // held them.  First -> second -> now in us: X = 2048, Y = 1536, the last 16 of 32 experts empty, 3000 rows in each
  // other 300 -> 301 -> 247, 28 empty and 4096 rows 181 -> 154 -> 148; X = Y = 1024, 56 of 64 empty, 3584 rows 117 -> 100 ->
  // 95; X = Y = 512, every second of 96 empty, 1200 rows 64 -> 65 -> 67.
  // In front of the loop the zeros held up its first tile, and between its tiles they cost the loop registers (65536
  // tokens, D = 4096, H = 2048, Wl1 gradient: 14.7 -> 15.1 ms).
  auto no_rows = [](const WTile& t) { return t.rows.re <= t.rows.rb && (!CUT || t.slot < 0); };
  auto next_tile = [&] {
    WTile t;
    do {
      t = items.next();
    } while (t.valid && no_rows(t));
    if (t.valid) place_tile(p, t), t.rows.forget_if_empty();
    return t;
  };

  auto zero_tiles = [&] {
    if (!items.some_empty) return;
    for (int at = blockIdx.x; at < p.N * items.tpe; at += gridDim.x) {
      WTile t;
      t.expert = at / items.tpe;
      t.q = at - t.expert * items.tpe;
      if (min(load_uniform(p.cumsums + t.expert + 1), p.msum) > min(load_uniform(p.cumsums + t.expert), p.msum)) continue;
      place_tile(p, t);
      zero_gw_tile(p, t);
    }
  };

  WTile c0 = next_tile();
  if (!c0.valid) {
    zero_tiles();
    trace.finish();
    return;
  }
  bf16* const lds = dyn_lds();
  constexpr int ELEMS = AOp::ELEMS;
  static_assert(ELEMS == BOp::ELEMS && 5 * ELEMS * sizeof(bf16) == kSpanLds, "three stages of B, two of A");
  const uint32_t addr = lds_address(lds);
  auto bslot = [&](int s) { return addr + (uint32_t)s * (ELEMS * 2) + BOp::wave_offset(); };
  auto aslot = [&](int s) { return addr + (uint32_t)(3 + s) * (ELEMS * 2) + AOp::wave_offset(); };
  auto bptr = [&](int s) { return (const bf16*)lds + s * ELEMS; };
  auto aptr = [&](int s) { return (const bf16*)lds + (3 + s) * ELEMS; };
  auto next3 = [](int s) { return s == 2 ? 0 : s + 1; };

  AOp A(p.a, p.lda, p.ga);
  BOp B(p.b, p.ldb, p.gb);
  A.set_tile(p.a, c0.rows, c0.x0, p.X);
  B.set_tile(p.b, c0.rows, c0.y0, p.Y);
  A.restart(c0.rows);
  B.restart(c0.rows);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    A.request();
    B.request();
    A.begin(c0.rows, s);
    B.begin(c0.rows, s);
    unrolled<0, BOp::DEP>([&](auto D) {
      B.template prepare<decltype(D)::value>();
      B.template deposit<decltype(D)::value>(bslot(s));
    });
    unrolled<0, AOp::DEP>([&](auto D) {
      A.template prepare<decltype(D)::value>();
      A.template deposit<decltype(D)::value>(aslot(s));
    });
  }
  wait_vmcnt<AOp::DEP + BOp::DEP>();
  __builtin_amdgcn_s_barrier();
  order_fence();
  int sb = 0, sa = 0;  // slots of the stage at hand
  int togo = c0.rows.stages() - 2;  // stages of the span at hand whose loads have not been started
  bool behind = true;               // the loads for the deposits that come next have not
  while (true) {
    WTile c1 = next_tile();
    if (!c1.valid) c1.rows = c0.rows, c1.x0 = c0.x0, c1.y0 = c0.y0;  // requests past the last item repeat its first stages
    const int rows = c0.rows.re - c0.rows.rb, real = (rows + kSpan - 1) / kSpan, count = c0.rows.stages();
    bool in_next = false;  // the loads have gone on to the next item
    // the loads for the stage after those started; past the next item's end the next round makes up for it
    auto request_next = [&] {
      behind = togo == 0 && in_next;
      if (behind) return;
      if (togo == 0) {
        in_next = true;
        togo = c1.rows.stages();
        A.restart(c1.rows);
        B.restart(c1.rows);
      }
      --togo;
      A.request();
      B.request();
    };
    if (behind) request_next();
    TileAcc acc;
    SpanFrags<AOp, BOp, FN, FM> fr(wave_row(), wave_col());
    const bf16 *b = bptr(sb), *a = aptr(sa);
    fr.template read_all<0, 0>(b, a);
    order_fence();
    auto turn = [&] {
      wait_vmcnt<BOp::DEP>();
      wait_lgkm0();
      __builtin_amdgcn_s_barrier();
      order_fence();
    };
    Span from = c0.rows;  // the span of the stages being requested,
    int ft = 2;              // the one at hand
    // Scalar loads share the wait counter of the LDS reads, and the products wait for those at the start of
    // each half: the loads start behind the wait in the middle of a stage, when both operands have used up the
    // last ones, and have half a stage.  The scalar unit issues one instruction in four cycles, and between the
    // halves no product runs: with A's loads at a stage's end and some 60 instructions in that place instead
    // of 25, the Wl1 gradient of 65536 tokens (D = 4096, H = 2048, N = 64, K = 8) took 15.2 ms instead of 14.3.
    static_assert(AOp::DEP == BOp::DEP, "prepared together");
    auto stage = [&](auto FRESH) {
      const uint32_t bto = bslot(sb == 0 ? 2 : sb - 1), ato = aslot(sa);
      sb = next3(sb);
      sa ^= 1;
      const bf16 *nb = bptr(sb), *na = aptr(sa);
      B.begin(from, ft);
      fr.template multiply<0, 1, BOp::DEP, decltype(FRESH)::value>(acc, b, a, [&](auto D) {
        B.template prepare<decltype(D)::value>();
        B.template deposit<decltype(D)::value>(bto);
        A.template prepare<decltype(D)::value>();
      });
      turn();
      request_next();
      A.begin(from, ft);
      fr.template multiply<1, 0, AOp::DEP>(acc, nb, na, [&](auto D) { A.template deposit<decltype(D)::value>(ato); });
      ++ft;
      b = nb;
      a = na;
    };
    int t = 0, end = count - 2;
    auto request_next_item = [&] {
      end = count;
      from = c1.rows;
      ft = 0;
      A.set_tile(p.a, from, c1.x0, p.X);
      B.set_tile(p.b, from, c1.y0, p.Y);
    };
    if (end == 0) request_next_item();
    if (real > 1) {  // the first stage by itself: its products start from zero (run_span_tiles)
      stage(IntC<true>{});
      t = 1;
    } else {
#pragma unroll
      for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[f][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    while (true) {
      const int stop = min(end, real - 1);
#pragma unroll 1
      for (; t < stop; ++t) stage(IntC<false>{});
      if (end == count) break;
      request_next_item();  // from here on its stages are requested
    }
    // the item's last stage: its k-values past the last row are zeroed on the M side, a half without rows is
    // left out; then, with 64 rows or fewer, a stage without rows
    for (; t < count; ++t) {
      const int left = rows - t * kSpan;
      const uint32_t bto = bslot(sb == 0 ? 2 : sb - 1), ato = aslot(sa);
      sb = next3(sb);
      sa ^= 1;
      auto mask = [&](auto SET, int nvalid) {  // rows `nvalid` and up of a half do not exist
        constexpr int set = decltype(SET)::value;
        wait_lgkm0();
        const int n = nvalid - 8 * (fresh_lane() >> 4);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          u32x4 v = __builtin_bit_cast(u32x4, fr.af[set][i]);
#pragma unroll
          for (int d = 0; d < 4; ++d) v[d] &= n >= 2 * d + 2 ? 0xFFFFFFFFu : n == 2 * d + 1 ? 0x0000FFFFu : 0u;
          fr.af[set][i] = __builtin_bit_cast(bf16x8, v);
        }
        order_fence();
      };
      auto deposit_b = [&](auto D) {
        B.template prepare<decltype(D)::value>();
        B.template deposit<decltype(D)::value>(bto);
        A.template prepare<decltype(D)::value>();
      };
      B.begin(from, ft);
      if (left > 0) {
        if (left < kHalf) mask(IntC<0>{}, left);
        fr.template multiply<0, 1, BOp::DEP>(acc, b, a, deposit_b);
      } else {
        unrolled<0, BOp::DEP>(deposit_b);
      }
      turn();
      request_next();
      A.begin(from, ft);
      if (left > kHalf) {
        if (left < kSpan) mask(IntC<1>{}, left - kHalf);
        fr.template multiply<1, -1, AOp::DEP>(acc, b, a, [&](auto D) { A.template deposit<decltype(D)::value>(ato); });
      } else {
        unrolled<0, AOp::DEP>([&](auto D) { A.template deposit<decltype(D)::value>(ato); });
      }
      ++ft;
    }
    // staging: where the item's last stage of B was (run_span_tiles)
    bf16* const staging = lds + (sb == 0 ? 2 : sb - 1) * ELEMS;
    if (!CUT || c0.slot < 0) {
      keep_in_place(acc);
      store_gw_tile(p, acc, c0.expert, c0.x0, c0.y0, staging);
    } else {
      store_partial(p, acc, c0.slot);
    }
    if (!c1.valid) break;
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    c0 = c1;
  }
  wait_vmcnt<0>();  // no transfer may outlive the workgroup's LDS
  zero_tiles();
  trace.finish();
}

// LDS of the reduction: the prefix sums, then the waves' staging
__host__ __device__ constexpr size_t reduce_plan_bytes(int N) { return ((size_t)(N + 1) * 20 + 512 + 15) / 16 * 16; }
constexpr size_t kReduceStaging = kSpanWaves * kStagingElems * sizeof(bf16);

// Adds up the partial tiles of the experts that wgrad_kernel cut into pieces and stores the bf16
// result.  Bound by memory: a workgroup takes 16 of a wave's 128 rows at a time, so that 32 registers hold its
// sums and four workgroups a CU their loads in flight.
__global__ __launch_bounds__(kSpanThreads) void wgrad_reduce_kernel(WgradArgs p) {
  drop_rows_of_an_overflowed_routing(p);
  const int tpe = p.tiles_x * p.tiles_y;
  const Plan pl = build_plan<kSpanThreads>(p, tpe);
  const int units = pl.ctiles[p.N] * FM;
  bf16* const staging = (bf16*)((char*)dyn_lds() + reduce_plan_bytes(p.N));
  for (int u = blockIdx.x; u < units; u += gridDim.x) {
    const int t = u / FM, i = u % FM;
    int lo = 0, hi = p.N;  // ctiles[lo] <= t < ctiles[hi]; the last such lo is the cut expert
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (pl.ctiles[mid] <= t) lo = mid; else hi = mid;
    }
    lo = uniform(lo);
    const int q = uniform(t - pl.ctiles[lo]);
    const int splits = uniform((pl.slots[lo + 1] - pl.slots[lo]) / tpe), slot0 = uniform(pl.slots[lo]) + q;
    f32x4 acc[FN][1];
#pragma unroll
    for (int f = 0; f < FN; ++f) acc[f][0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int piece = 0; piece < splits; ++piece)
#pragma unroll
      for (int f = 0; f < FN; ++f) acc[f][0] += partial_piece(p.ws, slot0 + piece * tpe, f, i)[lane_id()];
    WTile at;
    at.q = q;
    place_tile(p, at);
    const int x = at.x0 + wave_row() + 16 * i;
    store_rows<true>(acc, staging, p.gw + (int64_t)lo * p.X * p.Y, x, p.X - x, p.Y, at.y0 + wave_col(), lane_id(),
                     [](int) { return 1.0f; });
  }
}

template <class AOp, class BOp>
int launch(const WgradArgs& a, bool can_cut, hipStream_t st) {
  static LdsLimit once, once_cut, once_reduce;
  if (!can_cut) return launch_span(wgrad_kernel<false, AOp, BOp>, a, once, st);
  const int status = launch_span(wgrad_kernel<true, AOp, BOp>, a, once_cut, st);
  if (status != MOMOE_OK) return status;
  const size_t lds = reduce_plan_bytes(a.N) + kReduceStaging;
  if (!allow_lds(wgrad_reduce_kernel, reduce_plan_bytes(kMaxWgradExperts) + kReduceStaging, once_reduce)) return MOMOE_ERR_LAUNCH;
  wgrad_reduce_kernel<<<4 * persistent_grid(), kSpanThreads, lds, st>>>(a);
  return launch_status();
}

}  // namespace span

// Which loop.  Where a workgroup has eight tiles or more (ten with a k-blocked operand) that of gemm_span.hpp from 192 rows
// per expert on average, with a k-blocked operand and fewer than 128 experts from 256; where there are no more tiles
// than workgroups, so that the largest expert decides, from 192; elsewhere from 288.  Below, an expert is a few stages, the last of which may be half empty, and the eight waves of the other start and store
// sooner; many tiles hide the start and most of the stores.  Between 256 and 400 rows the second line is a compromise:
// loads that are the same for every expert or spread as by a router without preferences lose up to a tenth, skewed ones,
// whose large experts hold most of the work, gain as much.  32 rows a stage -> 64 in us, spread | falling as rank^-0.5.
// Wl2 gradient, 8 tiles a workgroup (D = 2048, H = 1024, N = 64) 200 rows 111 -> 104 | 110 -> 109, 300 132 -> 124 | 134 -> 126,
// 512 193 -> 169 | 195 -> 176; 16 (N = 128) 200 rows 211 -> 206 | 218 -> 220, 512 374 -> 348 | 384 -> 371; 4 (4096, 2048, 8) 200
// rows 53 -> 59 | 54 -> 58, 280 65 -> 65 | 65 -> 66, 400 81 -> 77 | 83 -> 73; 1 (512, 256, 96) 200 rows 24 -> 26 | 64 -> 59,
// 320 26 -> 28 | 93 -> 83, 400 28 -> 30 | 103 -> 81; 96 tiles (128, 256, 96) of 236 rows, falling as rank^-1.8, 166 -> 104.  Wl1 gradient, 32 tiles (2048, 1024, 128) 200 rows 402 -> 378 | 396 ->
// 403, 240 447 -> 413 | 431 -> 420; (2048, 2048, 64) 192 361 -> 381; 20 (2176, 1152, 64) 200 rows 221 -> 220 | 224 -> 237, 512
// 417 -> 409 | 402 -> 423; 4 (1024, 512, 64) 176 rows 51 -> 60 | 65 -> 63, 280 68 -> 72 | 77 -> 73, 400 79 -> 83 | 102 -> 96.
inline bool takes_span_loop(int64_t msum, int64_t n, int64_t x, int64_t y, bool kblocked) {
  const int64_t tiles = cdiv64(x, BX) * cdiv64(y, BY) * n, grid = persistent_grid();
  const bool many = tiles >= (kblocked ? 10 : 8) * grid;
  return msum >= (tiles <= grid || (many && (!kblocked || n >= 128)) ? 192 : many ? 256 : 288) * n;
}

}  // namespace
}  // namespace momoe

using namespace momoe;

// The most partial tiles a launch can use: kSplitsPerWorkgroup per workgroup, and no more than
// the pieces of kMinChunk k-stages that the rows can be cut into.
extern "C" int64_t momoe_wgrad_workspace_bytes(int64_t N, int64_t X, int64_t Y, int64_t Msum) {
  if (N <= 0 || X <= 0 || Y <= 0 || Msum < 0) return -1;
  const int64_t tpe = cdiv64(X, BX) * cdiv64(Y, BY);
  const int64_t by_rows = tpe * (Msum / kBK + N) / kMinChunk;
  return std::min<int64_t>((int64_t)kSplitsPerWorkgroup * kMaxWorkgroups, by_rows) *
         MOMOE_WGRAD_PARTIAL_BYTES;
}

extern "C" int64_t momoe_padded_rows(int64_t Msum, int64_t N) {
  if (Msum < 0 || N < 0) return -1;
  return ((Msum + 31) & ~(int64_t)31) + 32 * N;
}

extern "C" int momoe_wgrad_stage_rows(int64_t N, int64_t X, int64_t Y, int64_t Msum, int b_layout) {
  if (N <= 0 || X <= 0 || Y <= 0 || Msum <= 0) return 0;
  return takes_span_loop(Msum, N, X, Y, b_layout == MOMOE_LAYOUT_KBLOCKED) ? kSpan : kBK;
}

extern "C" int momoe_wgrad(const void* A, int64_t lda, int a_layout, const int32_t* a_gather,
                           const void* B, int64_t ldb, int b_layout, const int32_t* b_gather,
                           const int32_t* cumsums_N1, void* GW_NXY, int64_t M, int64_t N,
                           int64_t X, int64_t Y, int64_t Msum, void* workspace,
                           int64_t workspace_bytes, void* stream) {
  if (!A || !B || !cumsums_N1 || !GW_NXY) return MOMOE_ERR_BAD_ARG;
  if (M <= 0 || N <= 0 || X <= 0 || Y <= 0 || Msum <= 0) return MOMOE_ERR_BAD_ARG;
  const bool at = a_layout == MOMOE_LAYOUT_TRANSPOSED, bt = b_layout == MOMOE_LAYOUT_TRANSPOSED;
  const bool bk = b_layout == MOMOE_LAYOUT_KBLOCKED;
  if ((!at && a_layout != MOMOE_LAYOUT_ROWS) || (!bt && !bk && b_layout != MOMOE_LAYOUT_ROWS))
    return MOMOE_ERR_BAD_ARG;
  if (at && (bt || bk)) return MOMOE_ERR_UNSUPPORTED;  // one operand at most in a special layout
  // k-blocked B: ldb = rows of the matrix; features in whole blocks; 8 blocks of a tile are
  // addressed with 32-bit byte offsets
  if (bk && (b_gather != nullptr || ldb < Msum || Y % 32 != 0 || 8 * ldb * 64 >= (1ll << 32)))
    return b_gather != nullptr || ldb < Msum ? MOMOE_ERR_BAD_ARG : MOMOE_ERR_UNSUPPORTED;
  const int64_t mpad = momoe_padded_rows(Msum, N);
  if (lda < X || (!bk && ldb < Y) || (at && a_gather != nullptr) || (bt && b_gather != nullptr))
    return MOMOE_ERR_BAD_ARG;
  if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace) || ((uintptr_t)workspace & 15))
    return MOMOE_ERR_BAD_ARG;
  if (X % 8 != 0 || Y % 8 != 0 || lda % 8 != 0 || (!bk && ldb % 8 != 0)) return MOMOE_ERR_UNSUPPORTED;
  if (((uintptr_t)A & 15) || ((uintptr_t)B & 15) || ((uintptr_t)GW_NXY & 7))
    return MOMOE_ERR_BAD_ARG;
  if (Msum >= (1ll << 31) || mpad >= (1ll << 31) || X > (1 << 20) || Y > (1 << 20))
    return MOMOE_ERR_UNSUPPORTED;
  // rows are addressed with 32-bit byte offsets from the matrix base (gathered: M rows) or from
  // the first row of an expert's piece (an expert holds a token at most once: at most M rows);
  // a transposed operand needs no such offsets (a stage is one contiguous block)
  if ((!at && M * lda * 2 >= (1ll << 32)) || (!bt && !bk && M * ldb * 2 >= (1ll << 32)))
    return MOMOE_ERR_UNSUPPORTED;
  const int tiles_x = (int)cdiv64(X, BX), tiles_y = (int)cdiv64(Y, BY);
  // the per-expert prefix sums live in LDS while the work is dealt out; work items are
  // counted in 32 bits (every expert has its tiles, the cut ones at most ws_tiles more)
  const int grid = persistent_grid();
  const int64_t ws_tiles = std::min<int64_t>(workspace_bytes / MOMOE_WGRAD_PARTIAL_BYTES,
                                             (int64_t)kSplitsPerWorkgroup * std::min(grid, kMaxWorkgroups));
  if (N > kMaxWgradExperts || (int64_t)tiles_x * tiles_y * N + ws_tiles >= (1ll << 31))
    return MOMOE_ERR_UNSUPPORTED;
  // The launch has at most Msum/kBK + N k-stages per output tile.  With pieces of at least kc
  // stages the cut experts make at most tpe * stages / kc partial tiles: kc is chosen so that
  // they fit the workspace.
  int kc = 0x7fffffff;
  if (ws_tiles > 0) {
    const int64_t stages = (int64_t)tiles_x * tiles_y * (Msum / kBK + N);
    kc = (int)std::min<int64_t>(0x7fffffff, std::max<int64_t>(kMinChunk, cdiv64(stages, ws_tiles)));
  }
  WgradArgs a{(const bf16*)A, lda, a_gather, (const bf16*)B, ldb, b_gather, cumsums_N1,
              (bf16*)GW_NXY, (float*)workspace, kc, (int)N, (int)X, (int)Y, tiles_x, tiles_y,
              (int)Msum, clock_trace_buffer()};
  // an expert holds at most M rows: if that is short of the cutting length, nothing is cut
  const bool can_cut = kc != 0x7fffffff && cdiv64(std::min(M, Msum), kBK) >= 2 * (int64_t)kc;
  hipStream_t st = (hipStream_t)stream;
  if (takes_span_loop(Msum, N, X, Y, bk)) {
    if (at) return span::launch<span::TransposedOperand, span::RowsOperand>(a, can_cut, st);
    if (bt) return span::launch<span::RowsOperand, span::TransposedOperand>(a, can_cut, st);
    if (bk) return span::launch<span::RowsOperand, span::BlockedRowsOperand>(a, can_cut, st);
    return span::launch<span::RowsOperand, span::RowsOperand>(a, can_cut, st);
  }
  if (at) return tile::launch<tile::TransposedOperand, tile::RowsOperand, 4, 2>(a, can_cut, st);
  if (bt) return tile::launch<tile::RowsOperand, tile::TransposedOperand, 2, 4>(a, can_cut, st);
  if (bk) return tile::launch<tile::RowsOperand, tile::BlockedRowsOperand, 4, 2>(a, can_cut, st);
  return tile::launch<tile::RowsOperand, tile::RowsOperand, 4, 2>(a, can_cut, st);
}

extern "C" int momoe_backward_tail_fits(int64_t M, int64_t D, int64_t H, int64_t N, int64_t Msum) {
  if (M <= 0 || D <= 0 || H <= 0 || N <= 0 || Msum <= 0 || D % kBK != 0 || H % kBK != 0 || N > kMaxWgradExperts) return 0;
  // no expert can be long enough to be cut, and what the three products read and write besides the weights is little: it is
  // all there at once
  if (M >= 2 * kMinChunk * kBK || Msum < M || D > (1 << 20) || H > (1 << 19)) return 0;
  const int64_t bytes = (Msum * (2 * H + D) + momoe_padded_rows(Msum, N) * H) * (int64_t)sizeof(bf16);
  if (bytes > kTailBytes || D * H * 4 >= (1ll << 32) || cdiv64(D, BX) * cdiv64(2 * H, BY) * N >= (1ll << 31)) return 0;
  return !takes_span_loop(Msum, N, D, 2 * H, true) && !takes_span_loop(Msum, N, H, D, false) && !takes_span_tiles(Msum, N, D, 2 * H);
}

extern "C" int momoe_backward_tail(const void* hsT_GH32, int64_t ld_hsT, const void* Gy_MD, const void* x_MD,
                                   const void* gz_blocked, const void* Wl1_ND2H, const int32_t* idx_Msum,
                                   const int32_t* cumsums_N1, const int32_t* tile_table, void* GW2_NHD, void* GW1_ND2H,
                                   void* gxs_MsumD, const float* gs_part, int64_t nparts, float* Gs_MN, int64_t M, int64_t D,
                                   int64_t H, int64_t N, int64_t Msum, void* stream) {
  for (const void* p : {hsT_GH32, Gy_MD, x_MD, gz_blocked, Wl1_ND2H, (const void*)GW2_NHD, (const void*)GW1_ND2H,
                        (const void*)gxs_MsumD})
    if (!p || ((uintptr_t)p & 15)) return MOMOE_ERR_BAD_ARG;
  if (!idx_Msum || !cumsums_N1 || !tile_table || ld_hsT < H || ld_hsT % 8 != 0) return MOMOE_ERR_BAD_ARG;
  if (Gs_MN != nullptr && (!gs_part || nparts <= 0)) return MOMOE_ERR_BAD_ARG;
  if (!momoe_backward_tail_fits(M, D, H, N, Msum)) return MOMOE_ERR_UNSUPPORTED;
  auto weight = [&](const void* a, int64_t lda, const int32_t* ga, const void* b, int64_t ldb, const int32_t* gb, void* gw, int64_t X,
                    int64_t Y) {
    return WgradArgs{(const bf16*)a, lda, ga, (const bf16*)b, ldb, gb, cumsums_N1, (bf16*)gw, nullptr, 0x7fffffff, (int)N, (int)X,
                     (int)Y, (int)cdiv64(X, BX), (int)cdiv64(Y, BY), (int)Msum, clock_trace_buffer()};
  };
  const tile::TailArgs a{weight(x_MD, D, idx_Msum, gz_blocked, Msum, nullptr, GW1_ND2H, D, 2 * H),
                         weight(hsT_GH32, ld_hsT, nullptr, Gy_MD, D, idx_Msum, GW2_NHD, H, D),
                         {(const bf16*)gz_blocked, (const bf16*)Wl1_ND2H, tile_table, (bf16*)gxs_MsumD, (int)D, (int)H, Msum,
                          clock_trace_buffer()},
                         {gs_part, (int)nparts, idx_Msum, cumsums_N1, Gs_MN, (int)M, (int)N, Msum},
                         3 * D * H * N * (int64_t)sizeof(bf16) >= kBeyondCache ? 2u : 1u};
  constexpr size_t lds = std::max(tile::kWgradLds, kDxNarrowLds);
  static LdsLimit once;
  if (!allow_lds(tile::backward_tail_kernel, lds, once)) return MOMOE_ERR_LAUNCH;
  // (as many workgroups in a row as a launch has, a multiple of 8: a part's are on the XCDs that they take themselves to be on)
  const dim3 grid(persistent_grid(), tile::kTailParts - (Gs_MN != nullptr ? 0 : 1));
  tile::backward_tail_kernel<<<grid, kThreads, lds, (hipStream_t)stream>>>(a);
  return launch_status();
}
