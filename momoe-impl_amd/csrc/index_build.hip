// Routing index build: expert histogram, prefix sums, sorted-row scatter and
// the device-side tile table.  Integer work, HBM/latency bound: the mask is read
// twice with coalesced loads, positions come from wavefront ballots.
//
// Decomposition: the [N, M] mask is cut into panels of 16 experts x 256 tokens;
// one workgroup (256 lanes = 256 tokens) owns a panel.
//   pass 1 (count):   per panel, tokens per expert (ballot + popcount) and set
//                     bits per token.
//   pass 2 (scan):    one workgroup: per-expert exclusive scan over panels,
//                     exclusive scan over experts (cumsums), tile table.
//   pass 3 (scatter): per panel, each set bit learns its sorted row
//                     (expert base + panel base + wave base + rank in ballot) and
//                     its slot (set bits of the token in earlier experts).
// Up to kPlaceCounts panel counts and kPlaceMaxExperts experts, passes 2 and 3 are one launch
// (index_place_kernel): every panel's workgroup sums the counts it needs by itself.
#include <mutex>

#include "common.hpp"

namespace momoe {
namespace {

constexpr int kPanelTokens = 256;
constexpr int kPanelExperts = 16;
constexpr int kMaxExperts = 4096;

// The 16 mask entries of token m in expert group g, as a bit set.  Loads are unconditional (row
// and column clamped into the matrix, the result masked afterwards): a load under a branch is
// waited for before the next one is issued, which made this function one memory latency PER
// ENTRY instead of one per group.
__device__ __forceinline__ uint32_t load_panel_bits(const int32_t* __restrict__ mask, int64_t sn,
                                                    int64_t sm, int M, int N, int g, int m) {
  const int32_t* col = mask + (int64_t)min(m, M - 1) * sm;
  int32_t v[kPanelExperts];
#pragma unroll
  for (int e = 0; e < kPanelExperts; ++e)
    v[e] = col[(int64_t)min(g * kPanelExperts + e, N - 1) * sn];
  uint32_t bits = 0;
#pragma unroll
  for (int e = 0; e < kPanelExperts; ++e)
    bits |= (v[e] != 0 && g * kPanelExperts + e < N ? 1u : 0u) << e;
  return m < M ? bits : 0u;
}

__global__ __launch_bounds__(kPanelTokens) void index_count_kernel(
    const int32_t* __restrict__ mask, int64_t sn, int64_t sm, int M, int N,
    int32_t* __restrict__ part /*(expert i, panel c) at i * pn + c * pc*/, int pn, int pc,
    int32_t* __restrict__ tokcnt /*[NG][M]*/) {
  __shared__ int32_t wcnt[kPanelExperts][4];
  const int c = blockIdx.x, g = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int m = c * kPanelTokens + t;
  const uint32_t bits = load_panel_bits(mask, sn, sm, M, N, g, m);
#pragma unroll
  for (int e = 0; e < kPanelExperts; ++e) {
    const uint64_t b = __ballot((bits >> e) & 1u);
    if (lane == 0) wcnt[e][wave] = __popcll(b);
  }
  if (m < M) tokcnt[(int64_t)g * M + m] = __popc(bits);
  __syncthreads();
  if (t < kPanelExperts) {
    const int i = g * kPanelExperts + t;
    if (i < N) part[(int64_t)i * pn + (int64_t)c * pc] = wcnt[t][0] + wcnt[t][1] + wcnt[t][2] + wcnt[t][3];
  }
}

__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}

// Tile height for a routing (tile_rows = 0 asked for it).  A row tile streams its rows and a
// 256-column block of the expert's weights, so a GEMM's time goes with the sum over the tiles of
// (rows + 256): an expert of v rows costs v + 256 * (number of its tiles).  Tall tiles save whole
// passes over the weights (an expert of 513..640 rows: two instead of three) but their kernels
// are a few percent less efficient per tile: they are taken when they save more than 4 %.
__device__ __forceinline__ int choose_tile_rows(const int32_t* sizes, int N, int lane) {
  int64_t c_std = 0, c_tall = 0;
  for (int i = lane; i < N; i += 64) {
    const int v = sizes[i];
    c_std += v + 256 * ((v + MOMOE_RECOMPUTE_TILE_ROWS - 1) / MOMOE_RECOMPUTE_TILE_ROWS);
    c_tall += v + 256 * ((v + MOMOE_TILE_ROWS - 1) / MOMOE_TILE_ROWS);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    c_std += __shfl_xor(c_std, o);
    c_tall += __shfl_xor(c_tall, o);
  }
  return c_tall * 26 < c_std * 25 ? MOMOE_TILE_ROWS : MOMOE_RECOMPUTE_TILE_ROWS;
}

__global__ __launch_bounds__(1024) void index_scan_kernel(
    int32_t* __restrict__ part, int N, int NC, int64_t msum_cap,
    int64_t* __restrict__ sizes, int32_t* __restrict__ cumsums,
    int32_t* __restrict__ table, int tile_rows_arg, int32_t* __restrict__ table_rc,
    int32_t* __restrict__ violations, int32_t* __restrict__ idx, int32_t* __restrict__ which) {
  __shared__ int32_t s_size[kMaxExperts];
  __shared__ int32_t s_cum[kMaxExperts];
  __shared__ int32_t s_first[kMaxExperts];
  __shared__ int32_t s_total[3];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // per expert: exclusive scan of the panel counts, in place
  for (int i = wave; i < N; i += 16) {
    int running = 0;
    for (int c0 = 0; c0 < NC; c0 += 64) {
      const int c = c0 + lane;
      const int v = c < NC ? part[(int64_t)i * NC + c] : 0;
      const int inc = wave_inclusive_scan(v, lane);
      if (c < NC) part[(int64_t)i * NC + c] = running + inc - v;
      running += __shfl(inc, 63);
    }
    if (lane == 0) s_size[i] = running;
  }
  __syncthreads();
  if (wave == 0) {
    const int tile_rows = tile_rows_arg > 0 ? tile_rows_arg : choose_tile_rows(s_size, N, lane);
    int run_rows = 0, run_tiles = 0;
    for (int i0 = 0; i0 < N; i0 += 64) {
      const int i = i0 + lane;
      const int v = i < N ? s_size[i] : 0;
      const int nt = (v + tile_rows - 1) / tile_rows;
      const int inc = wave_inclusive_scan(v, lane);
      const int inct = wave_inclusive_scan(nt, lane);
      if (i < N) {
        s_cum[i] = run_rows + inc - v;
        s_first[i] = run_tiles + inct - nt;
        cumsums[i] = run_rows + inc - v;
        sizes[i] = (int64_t)v;
      }
      run_rows += __shfl(inc, 63);
      run_tiles += __shfl(inct, 63);
    }
    if (lane == 0) {
      cumsums[N] = run_rows;
      const bool overflow = (int64_t)run_rows > msum_cap;
      if (overflow) atomicAdd(violations, 1);
      s_total[0] = overflow ? 0 : run_tiles;
      s_total[1] = run_rows;
      s_total[2] = tile_rows;
      table[0] = overflow ? 0 : run_tiles;
      table[1] = tile_rows;
      table[2] = 0;
      table[3] = 0;
    }
  }
  __syncthreads();
  // A routing with fewer than M*K pairs leaves the sorted rows past the last pair without a
  // token: give them token 0 / slot 0, so that nothing downstream reads an undefined id.
  for (int64_t r = (int64_t)s_total[1] + t; r < msum_cap; r += 1024) {
    idx[r] = 0;
    which[r] = 0;
  }
  const int tile_rows = s_total[2];
  // the second table (tiles of the recomputing GEMM's height) is the same table when that is the
  // height chosen; otherwise the row tiles are counted again below
  const bool same = tile_rows == MOMOE_RECOMPUTE_TILE_ROWS;
  if (s_total[0] == 0) {
    if (table_rc != nullptr && t < kTileHeader) table_rc[t] = t == 1 ? MOMOE_RECOMPUTE_TILE_ROWS : 0;
    return;
  }
  auto write_entries = [&](int32_t* dst, int rows) {
    for (int i = t; i < N; i += 1024) {
      const int v = s_size[i];
      const int nt = (v + rows - 1) / rows;
      const int first = s_first[i];
      for (int k = 0; k < nt; ++k) {
        int32_t* e = dst + kTileHeader + 4 * (first + k);
        e[0] = i;
        e[1] = first;
        e[2] = s_cum[i];
        e[3] = v;
      }
    }
  };
  write_entries(table, tile_rows);
  if (table_rc == nullptr) return;
  if (same) {
    write_entries(table_rc, tile_rows);
    if (t < kTileHeader) table_rc[t] = t == 0 ? s_total[0] : t == 1 ? tile_rows : 0;
    return;
  }
  __syncthreads();  // every thread has read s_first
  if (wave == 0) {
    int run_tiles = 0;
    for (int i0 = 0; i0 < N; i0 += 64) {
      const int i = i0 + lane;
      const int v = i < N ? s_size[i] : 0;
      const int nt = (v + MOMOE_RECOMPUTE_TILE_ROWS - 1) / MOMOE_RECOMPUTE_TILE_ROWS;
      const int inct = wave_inclusive_scan(nt, lane);
      if (i < N) s_first[i] = run_tiles + inct - nt;
      run_tiles += __shfl(inct, 63);
    }
    if (lane < kTileHeader) table_rc[lane] = lane == 0 ? run_tiles : lane == 1 ? MOMOE_RECOMPUTE_TILE_ROWS : 0;
  }
  __syncthreads();
  write_entries(table_rc, MOMOE_RECOMPUTE_TILE_ROWS);
}

__global__ __launch_bounds__(kPanelTokens) void index_scatter_kernel(
    const int32_t* __restrict__ mask, int64_t sn, int64_t sm, int M, int N, int K, int NC,
    const int32_t* __restrict__ part, const int32_t* __restrict__ tokcnt,
    const int32_t* __restrict__ cumsums, int32_t* __restrict__ idx, int32_t* __restrict__ which,
    int32_t* __restrict__ inv, int32_t* __restrict__ violations) {
  __shared__ int32_t wcnt[kPanelExperts][4];
  const int c = blockIdx.x, g = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int m = c * kPanelTokens + t;
  const int64_t msum = (int64_t)M * K;
  const bool overflow = (int64_t)cumsums[N] > msum;
  const uint32_t bits = load_panel_bits(mask, sn, sm, M, N, g, m);
  uint64_t ballots[kPanelExperts];
#pragma unroll
  for (int e = 0; e < kPanelExperts; ++e) {
    ballots[e] = __ballot((bits >> e) & 1u);
    if (lane == 0) wcnt[e][wave] = __popcll(ballots[e]);
  }
  int k = 0;
  if (m < M)
    for (int gg = 0; gg < g; ++gg) k += tokcnt[(int64_t)gg * M + m];
  __syncthreads();
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int e = 0; e < kPanelExperts; ++e) {
    const int i = g * kPanelExperts + e;
    if (i >= N) break;
    if ((bits >> e) & 1u) {
      int woff = 0;
      for (int w = 0; w < wave; ++w) woff += wcnt[e][w];
      const int64_t row = (int64_t)cumsums[i] + part[(int64_t)i * NC + c] + woff +
                          __popcll(ballots[e] & below);
      if (row < msum) {
        idx[row] = m;
        which[row] = k;
      }
      // more pairs than rows: the GEMMs get an empty tile table and write nothing, so no token
      // may point at a row (the combine then gives zeros instead of unwritten memory)
      if (k < K) inv[(int64_t)m * K + k] = row < msum && !overflow ? (int32_t)row : -1;
      ++k;
    }
  }
  if (m < M && g == gridDim.y - 1 && k != K) {
    atomicAdd(violations, 1);
    // slots the token does not fill: -1 = "no row" (momoe_combine skips them)
    for (int kk = k; kk < K; ++kk) inv[(int64_t)m * K + kk] = -1;
  }
}

// one tile's entry, all of an expert's entries, and the header, in a table and (if asked for) in
// its copy for the recomputing GEMM
__device__ __forceinline__ void write_tile_entry(int32_t* table, int32_t* table_rc, int tile, int first,
                                                 int expert, int row0, int rows) {
  int32_t* e = table + kTileHeader + 4 * tile;
  e[0] = expert;
  e[1] = first;
  e[2] = row0;
  e[3] = rows;
  if (table_rc != nullptr) {
    int32_t* c = table_rc + kTileHeader + 4 * tile;
    c[0] = expert;
    c[1] = first;
    c[2] = row0;
    c[3] = rows;
  }
}
__device__ __forceinline__ void write_tile_entries(int32_t* table, int32_t* table_rc, int first,
                                                   int nt, int expert, int row0, int rows) {
  for (int k = 0; k < nt; ++k) write_tile_entry(table, table_rc, first + k, first, expert, row0, rows);
}
__device__ __forceinline__ void write_tile_header(int32_t* table, int32_t* table_rc, int ntiles,
                                                  int tile_rows) {
  table[0] = ntiles;
  table[1] = tile_rows;
  table[2] = 0;
  table[3] = 0;
  if (table_rc != nullptr) {
    table_rc[0] = ntiles;
    table_rc[1] = tile_rows;
    table_rc[2] = 0;
    table_rc[3] = 0;
  }
}

// The whole index build in one launch of one workgroup, for at most 64 tokens and 256 experts:
// thread e is EXPERT e and holds its row of the mask as a 64-bit set of tokens.  Transposing the
// mask costs one ballot per token (at most 64), a thread loads M mask entries, and an expert has
// its few rows placed in as many rounds: 4.8 us at 16 tokens x 128 experts.  (With a thread per
// token one workgroup can build up to 256 tokens' index, but it loads N entries per thread and
// needs N ballots: 15 us at 131 tokens, where counting and placing in two launches take 11.)
// MCH = ceil(M / 16): all of a thread's mask loads are in flight at once.
constexpr int kTinyTokens = 64;
template <int MCH>
__global__ __launch_bounds__(kPanelTokens) void index_tiny_kernel(
    const int32_t* __restrict__ mask, int64_t sn, int64_t sm, int M, int N, int K,
    int64_t* __restrict__ sizes, int32_t* __restrict__ cumsums, int32_t* __restrict__ idx,
    int32_t* __restrict__ which, int32_t* __restrict__ inv, int32_t* __restrict__ table,
    int tile_rows_arg, int32_t* __restrict__ table_rc, int32_t* __restrict__ violations,
    bool rows_of_int4) {
  static_assert(MCH >= 1 && 16 * MCH <= kTinyTokens, "token chunks of 16");
  const int tile_rows = tile_rows_arg > 0 ? tile_rows_arg : MOMOE_RECOMPUTE_TILE_ROWS;
  __shared__ uint64_t tokb[kTinyTokens][4];  // experts of token m among the experts of wave w, as a lane mask
  __shared__ int32_t s_slot[kTinyTokens][4];  // pairs of token m held by the experts of the waves below w
  __shared__ int32_t s_wave[4][2];
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
  const int64_t msum = (int64_t)M * K;
  // the expert's row of the mask as a bit set; loads unconditional, row and column clamped
  uint64_t bits = 0;
  const int32_t* row = mask + (int64_t)min(e, N - 1) * sn;
  if (rows_of_int4) {
    // contiguous rows of a multiple of 4 tokens, 16-byte aligned (checked on the host): four
    // tokens per load.  Lanes read rows that lie apart, so a load instruction costs one line
    // request per lane whatever its width, and this path makes a quarter of them.
    int4 v[4 * MCH];
#pragma unroll
    for (int c = 0; c < 4 * MCH; ++c) v[c] = ((const int4*)row)[min(c, M / 4 - 1)];
#pragma unroll
    for (int c = 0; c < 4 * MCH; ++c) {
      const uint64_t nib = (v[c].x != 0 ? 1u : 0u) | (v[c].y != 0 ? 2u : 0u) | (v[c].z != 0 ? 4u : 0u) |
                           (v[c].w != 0 ? 8u : 0u);
      if (4 * c < M) bits |= nib << (4 * c);
    }
  } else {
    int32_t v[16 * MCH];
#pragma unroll
    for (int m = 0; m < 16 * MCH; ++m) v[m] = row[(int64_t)min(m, M - 1) * sm];
#pragma unroll
    for (int m = 0; m < 16 * MCH; ++m) bits |= (uint64_t)(v[m] != 0 && m < M ? 1 : 0) << m;
  }
  if (e >= N) bits = 0;
  // per token: the experts that hold it
  for (int m = 0; m < M; ++m) {
    const uint64_t b = __ballot((bits >> m) & 1ull);
    if (lane == 0) tokb[m][wave] = b;
  }
  // exclusive scan over the experts of (rows, row tiles)
  const int v = __popcll(bits);
  const int nt = (v + tile_rows - 1) / tile_rows;
  const int irows = wave_inclusive_scan(v, lane), itiles = wave_inclusive_scan(nt, lane);
  if (lane == 63) {
    s_wave[wave][0] = irows;
    s_wave[wave][1] = itiles;
  }
  __syncthreads();
  int brow = irows - v, btile = itiles - nt;
  for (int w = 0; w < wave; ++w) {
    brow += s_wave[w][0];
    btile += s_wave[w][1];
  }
  const int total = s_wave[0][0] + s_wave[1][0] + s_wave[2][0] + s_wave[3][0];
  const int total_tiles = s_wave[0][1] + s_wave[1][1] + s_wave[2][1] + s_wave[3][1];
  const bool overflow = (int64_t)total > msum;
  if (e < N) {
    cumsums[e] = brow;
    sizes[e] = (int64_t)v;
    if (!overflow) write_tile_entries(table, table_rc, btile, nt, e, brow, v);
  }
  if (e == 0) {
    cumsums[N] = total;
    if (overflow) atomicAdd(violations, 1);
    write_tile_header(table, table_rc, overflow ? 0 : total_tiles, tile_rows);
  }
  // sorted rows past the last pair (a routing with fewer than M*K pairs): token 0, slot 0
  for (int64_t r = (int64_t)total + e; r < msum; r += kPanelTokens) {
    idx[r] = 0;
    which[r] = 0;
  }
  // thread m counts the pairs of token m
  int pairs = 0;
  if (e < M) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      s_slot[e][w] = pairs;
      pairs += __popcll(tokb[e][w]);
    }
  }
  __syncthreads();
  // the expert places its pairs, lowest token first; the slot of a pair within its token is the
  // number of lower-numbered experts that hold the token
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  uint64_t rest = bits;
  for (int r = 0; rest != 0; ++r) {
    const int m = __ffsll((unsigned long long)rest) - 1;
    rest &= rest - 1;
    const int k = s_slot[m][wave] + __popcll(tokb[m][wave] & below);
    const int64_t srow = (int64_t)brow + r;
    if (srow < msum) {
      idx[srow] = m;
      which[srow] = k;
    }
    if (k < K) inv[(int64_t)m * K + k] = srow < msum && !overflow ? (int32_t)srow : -1;
  }
  // tokens whose pair count is not K: thread m looks after token m
  if (e < M && pairs != K) {
    atomicAdd(violations, 1);
    for (int kk = pairs; kk < K; ++kk) inv[(int64_t)e * K + kk] = -1;
  }
}

// Results of all 64 lanes by the vector unit's lane permutations (quads, rows of 16, then from row to row), as uniform values
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t from_lanes(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, Op op) {  // op(v, 0) = v
  v = op(v, from_lanes<0xB1, 0xf>(v));   // quad_perm: lane ^ 1
  v = op(v, from_lanes<0x4E, 0xf>(v));   // quad_perm: lane ^ 2
  v = op(v, from_lanes<0x141, 0xf>(v));  // row_half_mirror: the other quad of 8 lanes
  v = op(v, from_lanes<0x140, 0xf>(v));  // row_mirror: the other half of 16 lanes
  v = op(v, from_lanes<0x142, 0xa>(v));  // row_bcast15: row 0 -> 1, row 2 -> 3
  v = op(v, from_lanes<0x143, 0xc>(v));  // row_bcast31: row 1 -> 2, 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The whole index build in one launch for one panel of tokens, at most 256, at most kColumnExperts experts and tiles of at
// least 256 rows (an expert is one tile): a workgroup per group of 16 experts, a thread per token.  Each reads the
// whole mask, all of a thread's entries in flight together, so that it knows by itself the pairs and tiles of the groups
// before its own; a launch that counts first takes longer.  Bound by the latency of the loads and of the exchanges between
// the waves.  In a graph, us with one fill of 1.6 us, counting and placing -> this: 128 tokens x 8 experts 8.9 -> 7.0,
// 200 x 64 10.1 -> 8.4; with a second round of loads, 131 x 128 10.2 -> 10.2, and a fourth, 256 x 256, 10.6 -> 14.7: up to 64
// experts.  The kernel above -> this: 64 x 8 10.4 -> 7.0, 64 x 64 9.0 -> 7.9, 48 x 64 8.2 -> 7.9, 32 x 64 7.1 -> 7.9: from
// more than kTinyFewExperts tokens on.
constexpr int kColumnExperts = 64, kTinyFewExperts = 48;
__global__ __launch_bounds__(kPanelTokens) void index_column_kernel(
    const int32_t* __restrict__ mask, int64_t sn, int64_t sm, int M, int N, int K, int NG, int64_t* __restrict__ sizes,
    int32_t* __restrict__ cumsums, int32_t* __restrict__ idx, int32_t* __restrict__ which, int32_t* __restrict__ inv,
    int32_t* __restrict__ table, int tile_rows, int32_t* __restrict__ table_rc, int32_t* __restrict__ violations) {
  constexpr int WAVES = kPanelTokens / 64, GROUPS = kColumnExperts / kPanelExperts;
  __shared__ uint32_t s_held[WAVES][GROUPS / 2];  // experts that hold a token of the wave, two groups a word
  __shared__ uint32_t s_pairs[WAVES];
  __shared__ int32_t s_off[kPanelExperts][WAVES];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, g = blockIdx.x, m = t;
  const int64_t msum = (int64_t)M * K;
  // a uniform row and the lane's 32-bit offset in it (checked on the host); clamped into the matrix, masked afterwards
  const uint32_t off = (uint32_t)min(m, M - 1) * (uint32_t)sm * 4;
  int32_t v[kColumnExperts];
#pragma unroll
  for (int e = 0; e < kColumnExperts; ++e) v[e] = *(const int32_t*)((const char*)(mask + (int64_t)min(e, N - 1) * sn) + off);
  uint32_t b[GROUPS], bits = 0;
  int k = 0, pairs = 0;  // of the token: pairs in the groups before this one, in all
#pragma unroll
  for (int u = 0; u < GROUPS; ++u) {
    b[u] = 0;
#pragma unroll
    for (int e = 0; e < kPanelExperts; ++e) b[u] |= (v[u * kPanelExperts + e] != 0 ? 1u : 0u) << e;
    const int left = N - u * kPanelExperts;  // experts there are
    b[u] &= m < M && left > 0 ? 0xffffu >> (kPanelExperts - min(left, kPanelExperts)) : 0u;
    const int n = __popc(b[u]);
    pairs += n;
    k += u < g ? n : 0;
    bits = u == g ? b[u] : bits;
  }
#pragma unroll
  for (int u = 0; u < GROUPS; u += 2) {
    const uint32_t held = wave_reduce(b[u] | b[u + 1] << 16, [](uint32_t x, uint32_t y) { return x | y; });
    if (lane == 0) s_held[wave][u / 2] = held;
  }
  uint64_t ballots[kPanelExperts];
#pragma unroll
  for (int q = 0; q < kPanelExperts; ++q) ballots[q] = __ballot((bits >> q) & 1u);
  // (at most 64 x 64 pairs of a wave's tokens: both sums in one word)
  const uint32_t sums = wave_reduce((uint32_t)k | (uint32_t)pairs << 16, [](uint32_t x, uint32_t y) { return x + y; });
  if (lane == 0) {
    s_pairs[wave] = sums;
#pragma unroll
    for (int q = 0; q < kPanelExperts; ++q) s_off[q][wave] = __popcll(ballots[q]);
  }
  __syncthreads();
  int base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) base += s_pairs[w] & 0xffff, total += s_pairs[w] >> 16;
  const bool overflow = (int64_t)total > msum;
  if (wave == 0) {
    // lane q: tiles of group q, which are its experts with tokens
    uint32_t held = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) held |= s_held[w][min(lane, GROUPS - 1) / 2];
    const int tiles = lane < NG ? __popc((held >> (16 * (lane & 1))) & 0xffff) : 0;
    const int tiles_to = wave_inclusive_scan(tiles, lane);
    const int tiles_before = __shfl(tiles_to - tiles, g), all_tiles = __shfl(tiles_to, 63);
    // lane e: expert e of this group
    const int i = g * kPanelExperts + lane;
    const bool mine = lane < kPanelExperts && i < N;
    int rows = 0;
    if (mine)
#pragma unroll
      for (int w = 0; w < WAVES; ++w) rows += s_off[lane][w];
    int run = base + wave_inclusive_scan(rows, lane) - rows;
    const uint64_t some = __ballot(rows > 0);
    if (mine) {
      const int tile = tiles_before + __popcll(some & ((1ull << lane) - 1));
      sizes[i] = (int64_t)rows;
      cumsums[i] = run;
      if (rows > 0 && !overflow) write_tile_entry(table, table_rc, tile, tile, i, run, rows);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {  // sorted row of the expert's first token, per wavefront
        const int n = s_off[lane][w];
        s_off[lane][w] = run;
        run += n;
      }
    }
    if (g == NG - 1 && lane == 0) {
      cumsums[N] = total;
      if (overflow) atomicAdd(violations, 1);
      write_tile_header(table, table_rc, overflow ? 0 : all_tiles, tile_rows);
    }
  }
  __syncthreads();
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int q = 0; q < kPanelExperts; ++q) {
    if ((bits >> q) & 1u) {
      const int row = s_off[q][wave] + __popcll(ballots[q] & below);
      if (row < msum) {
        idx[row] = m;
        which[row] = k;
      }
      if (k < K) inv[(int64_t)m * K + k] = row < msum && !overflow ? row : -1;  // (as index_place_kernel)
      ++k;
    }
  }
  if (g == NG - 1) {
    // sorted rows past the last pair (a routing with fewer than M*K pairs): token 0, slot 0
    for (int64_t r = (int64_t)total + t; r < msum; r += kPanelTokens) {
      idx[r] = 0;
      which[r] = 0;
    }
    if (m < M && pairs != K) {
      atomicAdd(violations, 1);
      for (int kk = pairs; kk < K; ++kk) inv[(int64_t)m * K + kk] = -1;
    }
  }
}

// Passes 2 and 3 in one launch, for N <= kPlaceMaxExperts and N * NC <= kPlaceCounts.  Every
// workgroup needs the rows of all experts before its panel, i.e. sums over all the counts (at most
// 64 KiB, from L2): doing that in each of them takes less time than a one-workgroup launch in
// front.  The panel's mask, its tokens' earlier pairs and the first counts are loaded together,
// so that a workgroup waits for memory once or twice; bases come from LDS (read from memory
// under the branch on a mask bit, they were waited for expert by expert).  Workgroup 0 writes what
// does not belong to a panel: sizes, cumsums and the tile tables, tile by tile (a thread per
// expert wrote all tiles of a large expert alone).
// Measured at 128 experts: 1000 tokens 9.1 + 11.6 (scan, scatter) -> 7.5 us, 8192 tokens 9.7 + 13.9
// -> 8.3; 65536 tokens x 64 experts 15.6 + 14.8 -> 18.9, and a launch fewer.
// The line at 16384 counts: a workgroup's sums grow with the counts and there are as many
// workgroups as panels, so the traffic goes with their square: 64 MB at 65536 tokens x 64 experts.
constexpr int kPlaceMaxExperts = 256;
constexpr int kPlaceCounts = 16384;

__device__ __forceinline__ int last_not_above(const int32_t* a, int n, int v) {
  int lo = 0, hi = n;  // a[lo] <= v < a[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] <= v) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(kPanelTokens) void index_place_kernel(
    const int32_t* __restrict__ mask, int64_t sn, int64_t sm, int M, int N, int K, int NC, int NG,
    const int32_t* __restrict__ part /*[NC][N]*/, const int32_t* __restrict__ tokcnt,
    int64_t* __restrict__ sizes, int32_t* __restrict__ cumsums, int32_t* __restrict__ idx,
    int32_t* __restrict__ which, int32_t* __restrict__ inv, int32_t* __restrict__ table,
    int tile_rows_arg, int32_t* __restrict__ table_rc, int32_t* __restrict__ violations) {
  __shared__ int32_t s_tot[kPlaceMaxExperts], s_pre[kPlaceMaxExperts];  // [slice][expert]
  __shared__ int32_t s_cum[kPlaceMaxExperts], s_first[kPlaceMaxExperts];
  __shared__ int32_t s_wave[4], s_off[kPanelExperts][4], s_height;
  static_assert(kPlaceMaxExperts == kPanelTokens, "a thread per expert");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t msum = (int64_t)M * K;
  const bool writer = blockIdx.x == 0;
  const int panel = max((int)blockIdx.x - 1, 0);
  const int g = panel / NC, c = panel - g * NC;
  const int m = c * kPanelTokens + t;
  constexpr int kMaxGroups = kPlaceMaxExperts / kPanelExperts;
  // pairs of this token in the groups of experts before g
  int32_t cnt[kMaxGroups];
  uint32_t bits = 0;
  if (!writer) {
    const int32_t* tc = tokcnt + min(m, M - 1);
#pragma unroll
    for (int q = 0; q < kMaxGroups; ++q) cnt[q] = tc[(int64_t)min(q, g) * M];
    bits = load_panel_bits(mask, sn, sm, M, N, g, m);
  }
  // rows of every expert, and those in the panels before c: the panels are dealt to
  // 256 / (experts rounded up to a power of two) slices of threads
  int ep = 1;
  while (ep < N) ep <<= 1;
  const int e = t & (ep - 1), slice = t / ep, slices = kPanelTokens / ep;
  int tot = 0, pre = 0;
  for (int c0 = slice; c0 < NC; c0 += 16 * slices) {
    int32_t v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = part[(int64_t)min(c0 + q * slices, NC - 1) * N + min(e, N - 1)];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int cc = c0 + q * slices;
      tot += cc < NC ? v[q] : 0;
      pre += cc < min(c, NC) ? v[q] : 0;
    }
  }
  s_tot[t] = tot;
  s_pre[t] = pre;
  uint64_t ballots[kPanelExperts];
#pragma unroll
  for (int q = 0; q < kPanelExperts; ++q) ballots[q] = __ballot((bits >> q) & 1u);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < kPanelExperts; ++q) s_off[q][wave] = __popcll(ballots[q]);
  __syncthreads();
  int v = 0, before = 0;
  if (t < N)
    for (int q = 0; q < slices; ++q) {
      v += s_tot[q * ep + t];
      before += s_pre[q * ep + t];
    }
  const int inc = wave_inclusive_scan(v, lane);
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  int cum = inc - v;
  for (int w = 0; w < wave; ++w) cum += s_wave[w];
  const int total = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
  const bool overflow = (int64_t)total > msum;

  if (writer) {
    s_tot[t] = v;  // each thread has read its own column of the slices; others' are re-read below
    if (t < N) {
      cumsums[t] = cum;
      sizes[t] = (int64_t)v;
    }
    s_cum[t] = cum;
    if (t == 0) {
      cumsums[N] = total;
      if (overflow) atomicAdd(violations, 1);
    }
    // sorted rows past the last pair (a routing with fewer than M*K pairs): token 0, slot 0
    for (int64_t r = (int64_t)total + t; r < msum; r += kPanelTokens) {
      idx[r] = 0;
      which[r] = 0;
    }
    __syncthreads();
    if (wave == 0) {
      const int h = tile_rows_arg > 0 ? tile_rows_arg : choose_tile_rows(s_tot, N, lane);
      if (lane == 0) s_height = h;
    }
    __syncthreads();
    const int height = s_height;
    auto write_table = [&](int32_t* dst, int32_t* copy, int rows) {
      const int nt = (v + rows - 1) / rows;
      const int inct = wave_inclusive_scan(nt, lane);
      if (lane == 63) s_wave[wave] = inct;
      __syncthreads();
      int first = inct - nt;
      for (int w = 0; w < wave; ++w) first += s_wave[w];
      s_first[t] = first;
      const int ntiles = overflow ? 0 : s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
      __syncthreads();
      if (t == 0) write_tile_header(dst, copy, ntiles, rows);
      for (int j = t; j < ntiles; j += kPanelTokens) {
        // the last expert whose first tile is not after j is the one that has tiles
        const int i = last_not_above(s_first, N, j);
        write_tile_entry(dst, copy, j, s_first[i], i, s_cum[i], s_tot[i]);
      }
      __syncthreads();
    };
    const bool same = height == MOMOE_RECOMPUTE_TILE_ROWS;
    write_table(table, same ? table_rc : nullptr, height);
    if (table_rc != nullptr && !same) write_table(table_rc, nullptr, MOMOE_RECOMPUTE_TILE_ROWS);
    return;
  }

  // sorted row of the first token of each of the panel's experts, per wavefront
  s_cum[t] = cum + before;
  __syncthreads();
  if (t < kPanelExperts && g * kPanelExperts + t < N) {
    int run = s_cum[g * kPanelExperts + t];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int n = s_off[t][w];
      s_off[t][w] = run;
      run += n;
    }
  }
  __syncthreads();
  int k = 0;
#pragma unroll
  for (int q = 0; q < kMaxGroups; ++q) k += q < g ? cnt[q] : 0;
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int q = 0; q < kPanelExperts; ++q) {
    if ((bits >> q) & 1u) {
      const int row = s_off[q][wave] + __popcll(ballots[q] & below);
      if (row < msum) {
        idx[row] = m;
        which[row] = k;
      }
      // more pairs than rows: the GEMMs get an empty tile table and write nothing, so no token
      // may point at a row (the combine then gives zeros instead of unwritten memory)
      if (k < K) inv[(int64_t)m * K + k] = row < msum && !overflow ? row : -1;
      ++k;
    }
  }
  if (m < M && g == NG - 1 && k != K) {
    atomicAdd(violations, 1);
    // slots the token does not fill: -1 = "no row" (momoe_combine skips them)
    for (int kk = k; kk < K; ++kk) inv[(int64_t)m * K + kk] = -1;
  }
}

// A tile table for another tile height from the prefix sums of a finished index build.
__global__ __launch_bounds__(1024) void tile_table_kernel(const int32_t* __restrict__ cumsums, int N,
                                                          int64_t msum_cap, int tile_rows,
                                                          int32_t* __restrict__ table) {
  __shared__ int32_t s_first[kMaxExperts];
  __shared__ int32_t s_tiles;
  const int t = threadIdx.x, lane = t & 63;
  if (t < 64) {
    int run_tiles = 0;
    for (int i0 = 0; i0 < N; i0 += 64) {
      const int i = i0 + lane;
      const int v = i < N ? cumsums[i + 1] - cumsums[i] : 0;
      const int nt = (v + tile_rows - 1) / tile_rows;
      const int inct = wave_inclusive_scan(nt, lane);
      if (i < N) s_first[i] = run_tiles + inct - nt;
      run_tiles += __shfl(inct, 63);
    }
    if (lane == 0) {
      // an index build that found more pairs than rows emptied its table: so does this one
      const int ntiles = (int64_t)cumsums[N] > msum_cap ? 0 : run_tiles;
      s_tiles = ntiles;
      table[0] = ntiles;
      table[1] = tile_rows;
      table[2] = 0;
      table[3] = 0;
    }
  }
  __syncthreads();
  if (s_tiles == 0) return;
  for (int i = t; i < N; i += 1024) {
    const int c = cumsums[i], v = cumsums[i + 1] - c;
    const int nt = (v + tile_rows - 1) / tile_rows;
    const int first = s_first[i];
    for (int k = 0; k < nt; ++k) {
      int32_t* e = table + kTileHeader + 4 * (first + k);
      e[0] = i;
      e[1] = first;
      e[2] = c;
      e[3] = v;
    }
  }
}

}  // namespace
}  // namespace momoe

using namespace momoe;

// The GEMMs deal an expert's 32-row fragment rows to its ceil(rows / tile_rows) tiles: with a tile
// height below 32, or one that is not a whole number of fragment rows, there would be more tiles
// than fragment rows (tiles without rows, addressed past the expert's end) or tiles taller than
// the height the table promises.  No GEMM takes tiles above MOMOE_TILE_ROWS.
static bool tile_height_ok(int tile_rows) {
  return tile_rows >= 32 && tile_rows <= MOMOE_TILE_ROWS && tile_rows % 32 == 0;
}

extern "C" int momoe_tile_table_build(const int32_t* cumsums_N1, int64_t N, int64_t Msum,
                                      int tile_rows, int32_t* tile_table, void* stream) {
  if (!cumsums_N1 || !tile_table || N <= 0 || Msum <= 0 || tile_rows <= 0) return MOMOE_ERR_BAD_ARG;
  if (N > kMaxExperts || Msum >= (1ll << 31) || !tile_height_ok(tile_rows)) return MOMOE_ERR_UNSUPPORTED;
  tile_table_kernel<<<1, 1024, 0, (hipStream_t)stream>>>(cumsums_N1, (int)N, Msum, tile_rows, tile_table);
  return launch_status();
}

extern "C" int64_t momoe_tile_table_ints(int64_t M, int64_t N, int64_t K, int tile_rows) {
  if (M < 0 || N < 0 || K < 0 || tile_rows < 0) return -1;
  // 0 = the library chooses between two heights: room for the shorter one
  return kTileHeader + 4 * max_row_tiles(M * K, N, tile_rows > 0 ? tile_rows : MOMOE_RECOMPUTE_TILE_ROWS);
}

extern "C" int64_t momoe_index_workspace_bytes(int64_t M, int64_t N) {
  if (M < 0 || N < 0) return -1;
  const int64_t NC = cdiv64(M, kPanelTokens), NG = cdiv64(N, kPanelExperts);
  return (N * NC + NG * M) * (int64_t)sizeof(int32_t) + 256;
}

extern "C" int momoe_index_build(const int32_t* mask_NM, int64_t stride_n, int64_t stride_m,
                                 int64_t M, int64_t N, int64_t K, int64_t* sizes_N,
                                 int32_t* cumsums_N1, int32_t* idx_Msum, int32_t* which_Msum,
                                 int32_t* inv_MK, int32_t* tile_table, int tile_rows,
                                 int32_t* recompute_table, void* workspace,
                                 int64_t workspace_bytes, int32_t* violations, void* stream) {
  if (!mask_NM || !sizes_N || !cumsums_N1 || !idx_Msum || !which_Msum || !inv_MK || !tile_table ||
      !workspace || !violations)
    return MOMOE_ERR_BAD_ARG;
  if (M <= 0 || N <= 0 || K <= 0 || tile_rows < 0) return MOMOE_ERR_BAD_ARG;
  if (N > kMaxExperts || M * K >= (1ll << 31) || M >= (1ll << 30)) return MOMOE_ERR_UNSUPPORTED;
  if (tile_rows != 0 && !tile_height_ok(tile_rows)) return MOMOE_ERR_UNSUPPORTED;
  // the second table goes with the library's own choice of the height
  if (recompute_table != nullptr && tile_rows != 0) return MOMOE_ERR_BAD_ARG;
  if (workspace_bytes < momoe_index_workspace_bytes(M, N)) return MOMOE_ERR_BAD_ARG;
  const int NC = (int)cdiv64(M, kPanelTokens), NG = (int)cdiv64(N, kPanelExperts);
  if (NG > 65535) return MOMOE_ERR_UNSUPPORTED;
  int32_t* part = (int32_t*)workspace;
  int32_t* tokcnt = part + N * NC;
  hipStream_t st = (hipStream_t)stream;
  // an expert is one tile; offsets in a row of the mask fit 32 bits
  const bool one_column = NC == 1 && N <= kColumnExperts && (tile_rows == 0 || tile_rows >= MOMOE_RECOMPUTE_TILE_ROWS) &&
                          stride_m >= 0 && stride_m < (1 << 20);
  if (M <= (one_column ? kTinyFewExperts : kTinyTokens) && N <= kPanelTokens) {
    auto kernel = M <= 16 ? index_tiny_kernel<1> : M <= 32 ? index_tiny_kernel<2>
                : M <= 48 ? index_tiny_kernel<3> : index_tiny_kernel<4>;
    const bool rows_of_int4 = stride_m == 1 && stride_n % 4 == 0 && M % 4 == 0 && ((uintptr_t)mask_NM & 15) == 0;
    kernel<<<1, kPanelTokens, 0, st>>>(mask_NM, stride_n, stride_m, (int)M, (int)N, (int)K, sizes_N,
                                       cumsums_N1, idx_Msum, which_Msum, inv_MK, tile_table,
                                       tile_rows, recompute_table, violations, rows_of_int4);
    return launch_status();
  }
  if (one_column) {
    // (left to choose, the height is 256: no expert has more rows)
    index_column_kernel<<<NG, kPanelTokens, 0, st>>>(
        mask_NM, stride_n, stride_m, (int)M, (int)N, (int)K, NG, sizes_N, cumsums_N1, idx_Msum, which_Msum, inv_MK, tile_table,
        tile_rows != 0 ? tile_rows : MOMOE_RECOMPUTE_TILE_ROWS, recompute_table, violations);
    return launch_status();
  }
  dim3 grid(NC, NG);
  const bool place = N <= kPlaceMaxExperts && N * NC <= kPlaceCounts;
  index_count_kernel<<<grid, kPanelTokens, 0, st>>>(mask_NM, stride_n, stride_m, (int)M, (int)N, part,
                                                    place ? 1 : NC, place ? (int)N : 1, tokcnt);
  if (place) {
    index_place_kernel<<<(unsigned)(NC * NG + 1), kPanelTokens, 0, st>>>(
        mask_NM, stride_n, stride_m, (int)M, (int)N, (int)K, NC, NG, part, tokcnt, sizes_N, cumsums_N1,
        idx_Msum, which_Msum, inv_MK, tile_table, tile_rows, recompute_table, violations);
    return launch_status();
  }
  index_scan_kernel<<<1, 1024, 0, st>>>(part, (int)N, NC, M * K, sizes_N, cumsums_N1, tile_table,
                                        tile_rows, recompute_table, violations, idx_Msum,
                                        which_Msum);
  index_scatter_kernel<<<grid, kPanelTokens, 0, st>>>(mask_NM, stride_n, stride_m, (int)M, (int)N,
                                                      (int)K, NC, part, tokcnt, cumsums_N1,
                                                      idx_Msum, which_Msum, inv_MK, violations);
  return launch_status();
}

// ---- the same without a caller-provided workspace ------------------------------------------
// The panel counts live in a fixed array in device memory that is part of the library's code
// object: every GPU the library runs on holds its own copy, at its own address, until the
// process ends.  In host code the array's NAME is only a handle for the runtime, not a device
// address: the address is looked up once per device and kept; kernels and every other use of
// the array's memory take that pointer.
namespace {
constexpr int64_t kStaticScratchBytes = MOMOE_INDEX_STATIC_SCRATCH_BYTES;
__attribute__((used)) static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on device d, once looked up

int scratch_of_current_device(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return MOMOE_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      return MOMOE_ERR_LAUNCH;
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MOMOE_OK;
}
}  // namespace

extern "C" int momoe_index_build_static(const int32_t* mask_NM, int64_t stride_n, int64_t stride_m,
                                        int64_t M, int64_t N, int64_t K, int64_t* sizes_N,
                                        int32_t* cumsums_N1, int32_t* idx_Msum,
                                        int32_t* which_Msum, int32_t* inv_MK, int32_t* tile_table,
                                        int tile_rows, int32_t* recompute_table,
                                        int32_t* violations, void* stream) {
  if (M <= 0 || N <= 0) return MOMOE_ERR_BAD_ARG;
  // sizes beyond the fixed array are refused, never truncated
  if (momoe_index_workspace_bytes(M, N) > kStaticScratchBytes) return MOMOE_ERR_UNSUPPORTED;
  void* ws = nullptr;
  const int st = scratch_of_current_device(&ws);
  if (st != MOMOE_OK) return st;
  // Every word of the array that the scatter pass reads was written by the count pass of the
  // same call, so nothing has to be cleared between calls.
  return momoe_index_build(mask_NM, stride_n, stride_m, M, N, K, sizes_N, cumsums_N1, idx_Msum,
                           which_Msum, inv_MK, tile_table, tile_rows, recompute_table, ws,
                           kStaticScratchBytes, violations, stream);
}
