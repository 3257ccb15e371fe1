// Workgroup-level bf16 GEMM for gfx950 (CDNA4): 256 x 256 fp32 tiles, 64 k-values a stage.
//
// A workgroup of 4 wavefronts, one per SIMD with the SIMD's whole register file, computes a tile
// with v_mfma_f32_16x16x32_bf16; each wave owns 128 x 128 of it in 8 x 8 accumulators
// of 4 registers.  One workgroup per CU, persistent.
//
// What bounds such a loop on MI355X is energy: under sustained MFMA load the chip is power-limited and
// the shader clock falls until the power fits, so time follows what is spent on multiplications,
// LDS reads and transfers, and idle issue slots come on top.  Hence:
//   * 128 x 128 per wave: a wave reads 256 rows and columns of LDS for 16384 products per k, where
//     two waves per SIMD with 128 x 64 each read 384.
//   * the 16 x 16 x 32 MFMA: the same products at 2.0 PFLOP/s where 32 x 32 x 16 sustains 1.75 on
//     random operands.
//   * 64 k-values a stage: a row of a k-contiguous operand is a whole 128-byte line, asked for once
//     (with 32 k-values every line was asked for twice).
//   * a lone wave per SIMD hides nothing behind another wave, so everything is placed by hand: between
//     the MFMAs of one half of a stage (32 k-values) lie the fragment reads of the next half
//     and one operand's transfers, a few MFMAs apart; two register sets of fragments.
//   * the request stream runs on across tiles: the last two stages of a tile request the
//     first two of the next one, and nothing drains before the epilogue or refills after it.
// Uniform product of 131072 rows in 16 experts, K = N = 4096, N(0,1) x N(0,0.02) operands, harness of
// the loop alone, TFLOP/s: 8 waves with 32 x 32 x 16 and 32 k-values a stage 1022 -> 8 waves, 64
// k-values 1273 -> 4 waves 1229 -> 8 waves with 16 x 16 x 32 1293 -> 4 waves with 16 x 16 x 32 1393.
//
// LDS: a ring of stages for each operand, one deeper for the weights, which come from HBM where rows
// mostly come out of L2: 3 x 32 KiB and 2 x 32 KiB.
//
// Global memory goes straight to LDS with global_load_lds_dwordx4; every lane chooses its own 16
// bytes, so the LDS image is swizzled by permuting which piece a lane fetches, and the same freedom
// does all predication: what does not exist is pointed at something that does, masked at the store.
//
// The MFMA's first input is the weight-side fragment (16 columns), its second the row-side one
// (16 rows): a lane holds, for one tile row (lane%16), columns 4*(lane/16) .. +3.
#pragma once
#include <cmath>

#include "gemm_tile.hpp"

namespace momoe {

constexpr int kSpan = 64;                   // k-extent of a stage
constexpr int kHalf = 32;                   // k-extent of one MFMA and of the smallest contraction
constexpr int kSpanThreads = 256;
constexpr int kSpanWaves = kSpanThreads / 64;
constexpr size_t kSpanLds = 160 << 10;      // all of a CU's

template <int V>
struct IntC {
  static constexpr int value = V;
};
template <int I, int N, class F>
__device__ __forceinline__ void unrolled(F f) {
  if constexpr (I < N) {
    f(IntC<I>{});
    unrolled<I + 1, N>(f);
  }
}
__device__ __forceinline__ void order_fence() { __builtin_amdgcn_sched_barrier(0); }
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
// The lane, as a value of its own each time: what is derived from it is computed where it is used.  Taken
// from lane_id() in a tile's set-up or epilogue it would be hoisted out of the tile loop, and a main
// loop that owns every register has it spilled; each reload then waits for the stores before it
// (h.Wl2 with 1024 k-values: 449 us where 300 are due).
__device__ __forceinline__ int fresh_lane() {
  int l = lane_id();
  asm volatile("" : "+v"(l));
  return l;
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 first, bf16x8 second, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(first, second, c, 0, 0, 0);
}

// 16 bytes per lane, global -> LDS, as dma16; the LDS address is the sum of a scalar and a constant
template <int IMM>
__device__ __forceinline__ void dma16_at(const void* uniform_base, uint32_t byte_offset, uint32_t lds_wave_base) {
  asm volatile("s_add_u32 m0, %2, %3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(byte_offset), "s"(uniform_base),
               "s"(lds_wave_base), "n"(IMM)
               : "memory", "scc");
}

// Stores 16 bytes per lane at a uniform base plus a byte offset below 2 GiB; lanes that are not `valid` store
// nothing.  Without a branch: under a divergent one the compiler took what follows it for divergent, too.
// STREAM: non-temporal.
template <bool STREAM = false>
__device__ __forceinline__ void store16(void* uniform_base, uint32_t byte_offset, bool valid, bf16x8 v) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_base, 0, 0x7FFFFFFF, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, valid ? byte_offset : 0xFFFFFFF0u, 0, STREAM ? 2 : 0);
}

// The same with one bound for all lanes: those whose offset lies at or past `bytes`, a uniform value, store nothing.
// For a store that many are made of: the comparison costs no instructions.
template <bool STREAM = false>
__device__ __forceinline__ void store16_below(void* uniform_base, uint32_t byte_offset, uint32_t bytes, bf16x8 v) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_base, 0, bytes, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, byte_offset, 0, STREAM ? 2 : 0);
}
// how many of a fragment row's 16 rows, from `row` on, are among the first `rows` (a median is taken in vector registers)
__device__ __forceinline__ uint32_t rows_of_fragment(int row, int rows) {
  return __builtin_amdgcn_readfirstlane(max(0, min(16, rows - row)));
}

// the same for 4 bytes
__device__ __forceinline__ void store4(float* uniform_base, uint32_t byte_offset, bool valid, float v) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_base, 0, 0x7FFFFFFF, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc, valid ? byte_offset : 0xFFFFFFF0u, 0, 0);
}

// ---- operands -------------------------------------------------------------------------------------
// Common to all: DEP deposits (wave-wide transfers of 1 KiB) per wave and stage; source(k) is where the
// stage that starts at k-value k (a multiple of 32) lies, deposit<j>(source, slot) requests the j-th into
// the slot at LDS byte address slot - 1024 * wave; Lane(org) prepares the fragment reads of this lane for rows (columns) org.., frag(slot, lane, i, h) is the
// fragment of the 16 rows from org + 16 i, half h of the stage.

// Rows of 64 k-values, k-contiguous.  LDS [ROWS][64]: the 16-byte piece p of row r at position
// p ^ ((r / 2) % 8), so that the 16 rows x 16 bytes of 16 lanes of a fragment read cover all banks.
template <int ROWS>
struct SpanRowsLayout {
  static constexpr int DEP = ROWS / 32;
  // row that lane l fetches in the first deposit; the others lie 32 rows apart
  static __device__ __forceinline__ int first_row(int l) { return wave_id() * 8 + (l >> 3); }
  // piece of a row that it fetches (the same in every deposit), as a byte offset
  static __device__ __forceinline__ uint32_t piece_bytes(int l) { return ((l & 7) ^ ((first_row(l) >> 1) & 7)) * 16; }
  static constexpr int at(int j) { return j * kSpanWaves * 1024; }
  static constexpr int ELEMS = ROWS * kSpan;
  struct Lane {
    int o[2];  // bytes
    __device__ __forceinline__ explicit Lane(int org) {
      const int l = fresh_lane(), r = l & 15, g = l >> 4;
#pragma unroll
      for (int h = 0; h < 2; ++h) o[h] = (org + r) * (2 * kSpan) + ((4 * h + g) ^ (r >> 1)) * 16;
    }
  };
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) {
    return *(const bf16x8*)((const char*)slot + ln.o[h] + i * (32 * kSpan));
  }
};

// gathered rows: one byte offset per deposit
template <int ROWS>
struct SpanGatheredRows : SpanRowsLayout<ROWS> {
  using L = SpanRowsLayout<ROWS>;
  const bf16* base;
  uint32_t off[L::DEP];
  // rowbytes(j, l) = byte offset from base_ of the row that lane l fetches in deposit j
  template <class RowBytes>
  __device__ __forceinline__ void init(const bf16* base_, RowBytes rowbytes) {
    base = base_;
    const int l = fresh_lane();
    const uint32_t piece = L::piece_bytes(l);
#pragma unroll
    for (int j = 0; j < L::DEP; ++j) off[j] = rowbytes(j, l) + piece;
  }
  // nothing more will be needed: one line per deposit from here on
  __device__ __forceinline__ void idle() {
#pragma unroll
    for (int j = 0; j < L::DEP; ++j) off[j] = 0;
  }
  __device__ __forceinline__ const bf16* source(int k) const { return base + (uint32_t)k; }
  template <int j>
  __device__ __forceinline__ void deposit(const bf16* src, uint32_t slot) const {
    dma16_at<L::at(j)>(src, off[j], slot);
  }
};

// Rows at a fixed pitch (k-contiguous weights).  The matrix holds a multiple of 32 rows, and a deposit
// of the four waves covers 32: where the tile sticks out the last 32 are repeated.
template <int ROWS>
struct SpanPitchedRows : SpanRowsLayout<ROWS> {
  using L = SpanRowsLayout<ROWS>;
  const bf16* base;
  uint32_t off, pitch;  // bytes
  int last;             // first row, relative to the tile, of the matrix' last 32
  __device__ __forceinline__ void init(const bf16* mat, int K, int row0, int nrows) {
    pitch = (uint32_t)K * 2;
    base = mat + (int64_t)row0 * K;
    const int l = fresh_lane();
    off = (uint32_t)L::first_row(l) * pitch + L::piece_bytes(l);
    last = nrows - 32 - row0;
  }
  __device__ __forceinline__ void idle() { off = 0, last = 0; }
  __device__ __forceinline__ const bf16* source(int k) const { return base + (uint32_t)k; }
  template <int j>
  __device__ __forceinline__ void deposit(const bf16* src, uint32_t slot) const {
    dma16_at<L::at(j)>((const char*)src + (uint32_t)min(32 * j, last) * pitch, off, slot);
  }
};

// Sorted rows of a k-blocked matrix: element (row, k) at mat[((k / 32) * nrows + row) * 32 + k % 32].
// LDS [2][ROWS][32], each half as the matrix has it, piece p of row r at p ^ swz(r).
template <int ROWS>
struct SpanBlockedRows {
  // 0, 2, 3, 1 for consecutive groups of 4 rows: a 16-byte LDS read serves lanes 0-3, 12-15, 20-23 and
  // 24-27 in one clock, 4-11, 16-19 and 28-31 in the next; with r / 4 itself lanes 0-3 and 20-23 met
  // in the same banks (a third of the LDS' busy cycles)
  static __device__ __forceinline__ int swz(int r) { return ((r >> 2) & 1) * 2 ^ ((r >> 3) & 1) * 3; }
  static constexpr int DEP = ROWS / 32, PER_HALF = DEP / 2;
  static constexpr int ELEMS = ROWS * kSpan;
  const bf16* base;
  int64_t kstride;  // elements between k-blocks
  uint32_t off[PER_HALF];
  __device__ __forceinline__ void init(const bf16* mat, int64_t nrows, int64_t row0, int nvalid) {
    kstride = nrows * kHalf;
    base = mat + row0 * kHalf;
    const int l = fresh_lane();
#pragma unroll
    for (int j = 0; j < PER_HALF; ++j) {
      const int row = (j * kSpanWaves + wave_id()) * 16 + (l >> 2);
      off[j] = (uint32_t)min(row, nvalid - 1) * (kHalf * 2) + (((l & 3) ^ swz(row)) * 16);
    }
  }
  __device__ __forceinline__ void idle() {
#pragma unroll
    for (int j = 0; j < PER_HALF; ++j) off[j] = 0;
  }
  __device__ __forceinline__ const bf16* source(int k) const { return base + (int64_t)(k / kHalf) * kstride; }
  template <int j>
  __device__ __forceinline__ void deposit(const bf16* src, uint32_t slot) const {
    constexpr int h = j / PER_HALF, q = j % PER_HALF;
    dma16_at<h * (ROWS * kHalf * 2) + q * kSpanWaves * 1024>(h ? src + kstride : src, off[q], slot);
  }
  struct Lane {
    int o;
    __device__ __forceinline__ explicit Lane(int org) {
      const int l = fresh_lane(), r = l & 15, g = l >> 4;
      o = (org + r) * (2 * kHalf) + (g ^ swz(r)) * 16;
    }
  };
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) {
    return *(const bf16x8*)((const char*)slot + ln.o + h * (ROWS * kHalf * 2) + i * (32 * kHalf));
  }
};

// k-strided columns at a fixed pitch ([k][n] weights).  LDS [64][COLS]; the 16-byte piece p of k-row k at
// p ^ swz(k).  A fragment is two ds_read_b64_tr_b16, the LDS transpose read: within each group of 16
// lanes, lane i supplies the address of columns 4 * (i % 4) .. +3 of k-row i / 4 and receives column
// i of those 4 k-rows.  The 8 k-rows x 32 bytes of 32 lanes then lie in different banks.
// PAIRED: the wave's second half of fragments are the columns COLS / 2 further on.
template <bool PAIRED = false>
struct SpanCols {
  static constexpr int COLS = 256, DEP = COLS / 32, FN = COLS / 32;
  static constexpr int ELEMS = COLS * kSpan;
  static constexpr int PIECES = COLS / 8, RPD = 64 / PIECES;  // pieces of a k-row, k-rows of a deposit
  static constexpr int STEP = RPD * kSpanWaves;                // k-rows of a deposit of all waves
  static constexpr int PATTERNS = 2;                           // swizzles met by this lane's deposits
  static __device__ __forceinline__ int swz(int k) { return 2 * (k & 3) + 8 * ((k >> 3) & 1); }
  const bf16* base;
  uint32_t off[PATTERNS], pitch;  // bytes
  // coloff(c) = element offset from base_ of tile column c (a multiple of 8) of k-row 0, readable
  template <class ColOff>
  __device__ __forceinline__ void init(const bf16* base_, int ld, ColOff coloff) {
    base = base_;
    pitch = (uint32_t)ld * 2;
    const int l = fresh_lane(), krow = wave_id() * RPD + l / PIECES;
#pragma unroll
    for (int q = 0; q < PATTERNS; ++q)
      off[q] = (uint32_t)krow * pitch + (uint32_t)coloff(((l % PIECES) ^ swz(krow + STEP * q)) * 8) * 2;
  }
  __device__ __forceinline__ void idle() {
    pitch = 0;
#pragma unroll
    for (int q = 0; q < PATTERNS; ++q) off[q] = 0;
  }
  __device__ __forceinline__ const bf16* source(int k) const { return (const bf16*)((const char*)base + (uint32_t)k * pitch); }
  template <int j>
  __device__ __forceinline__ void deposit(const bf16* src, uint32_t slot) const {
    dma16_at<j * kSpanWaves * 1024>((const char*)src + (uint32_t)(STEP * j) * pitch, off[j % PATTERNS], slot);
  }
  struct Lane {
    int o;  // first fragment, in bytes
    __device__ __forceinline__ explicit Lane(int org) {
      const int l = fresh_lane(), krow = 8 * (l >> 4) + ((l & 15) >> 2), col = org + 4 * (l & 3);
      o = (krow * COLS + (((col >> 3) ^ swz(krow)) << 3) + (col & 7)) * 2;
    }
  };
  static __device__ __forceinline__ bf16x8 frag(const bf16* slot, const Lane& ln, int i, int h) {
    // (pieces 1 to 3 bits up are permuted, so what is added to a column there is an exclusive or)
    const int far = PAIRED && i >= FN / 2 ? COLS / 2 : 0, n = PAIRED ? i % (FN / 2) : i;
    const bf16* p = (const bf16*)((const char*)slot + (ln.o ^ (32 * n))) + far + h * (kHalf * COLS);
    const bf16x4 lo = lds_read_tr4(p), hi = lds_read_tr4(p + 4 * COLS);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// ---- tile geometries --------------------------------------------------------------------------------
// Waves 2 x 2, each 128 rows and 128 columns.
struct WideSpan {
  static constexpr int COLS = 256, MAX_ROWS = 256;
  static constexpr int AHEAD = 2;               // stages of rows in LDS; of weights one more
  static constexpr int FM = 8, FN = COLS / 32;  // 16-row and 16-column fragments of a wave
  static constexpr int WROWS = 2, WCOLS = 2;
};

// Tile order: that of TileSchedT (tables of taller tiles are halved) as long as an XCD has a tile for every
// workgroup.  What is left after its last full round, if that is at most half a round, is cut by its
// 32-row fragment rows into as many pieces, up to 8, as there are workgroups for, and every workgroup
// does one: without the cut a launch with 324 tiles for 256 CUs takes as long as one with 512.
template <class G>
struct SpanSched {
  using Tiles = TileSchedT<G::WROWS, G::MAX_ROWS, kSpanWaves>;
  struct Raw {
    typename Tiles::Raw tile;
    bool piece;
  };
  Tiles tiles;
  int rest, cut;  // tiles that are cut, into how many pieces (0: nothing left to do)
  __device__ __forceinline__ SpanSched(const int* table, int nb, int max_tile_rows, int first)
      : tiles(table, nb, max_tile_rows, first) {
    rest = tiles.limit % tiles.stride;
    cut = 8 * rest <= tiles.stride ? 8 : 4 * rest <= tiles.stride ? 4 : 2;
    if (2 * rest > tiles.stride || rest == 0) cut = 0;
    else tiles.limit -= rest;
  }
  __device__ __forceinline__ int order() const { return blockIdx.x >> 3; }  // of this workgroup in its XCD
  __device__ __forceinline__ Raw fetch() {
    const bool whole = tiles.pos < tiles.limit;
    Raw r;
    r.piece = !whole && cut > 0 && order() < rest * cut;
    r.tile = tiles.entry(whole ? tiles.pos : tiles.limit + order() / max(cut, 1), whole || r.piece);
    if (!whole) rest = 0;
    tiles.pos += tiles.stride;
    return r;
  }
  __device__ __forceinline__ TileCoord resolve(const Raw& r) const {
    TileCoord tc = tiles.resolve(r.tile);
    if (!r.piece || !tc.valid) return tc;
    const int nf = (tc.rows + 31) >> 5, part = order() % cut;
    const int base = nf / cut, extra = nf - base * cut, f0 = part * base + min(part, extra);
    tc.row0 += 32 * f0;
    tc.prow0 += 32 * f0;
    tc.rows = min(32 * (base + (part < extra ? 1 : 0)), tc.rows - 32 * f0);
    tc.valid = tc.rows > 0;
    Tiles::deal(tc);
    return tc;
  }
  __device__ __forceinline__ TileCoord next() { return resolve(fetch()); }
};

// ---- the k-loop -----------------------------------------------------------------------------------
// Stages of a contraction over K k-values, a multiple of 32 and at least 64 AHEAD.  The last one starts at
// K - 64 and is multiplied by its second half only where K is an odd multiple of 32.
struct SpanStages {
  int full, count, kmax;
  bool tail;
  __device__ __forceinline__ explicit SpanStages(int K)
      : full(K / kSpan), count((K + kSpan - 1) / kSpan), kmax(K - kSpan), tail(K % kSpan != 0) {}
  __device__ __forceinline__ int after(int k) const { return min(k + kSpan, kmax); }  // k-origin of the next stage
};

// Copies of the accumulators to vector registers are made after this point, where they are used: made ahead,
// beside a main loop's fragments, they were spilled, and every reload waits for the stores before it.
template <int FN, int NA>
__device__ __forceinline__ void keep_in_place(f32x4 (&acc)[FN][NA]) {
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < NA; ++i) asm volatile("" : "+a"(acc[j][i]));
}

// A wave's fragments of a stage, NA of rows and FN of weights, in two register sets
template <class Rows, class Weights, int FN, int NA>
struct SpanFrags {
  static constexpr int NM = NA * FN;
  typename Rows::Lane alane;
  typename Weights::Lane wlane;
  bf16x8 af[2][NA > 0 ? NA : 1], wf[2][FN];
  __device__ __forceinline__ SpanFrags(int m_org, int n_org) : alane(m_org), wlane(n_org) {}
  // fragment R (weights first) of half H of the stage at (w, a) into register set B
  template <int B, int R, int H>
  __device__ __forceinline__ void read(const bf16* w, const bf16* a) {
    if constexpr (NA == 0) return;
    else if constexpr (R < FN) wf[B][R] = Weights::frag(w, wlane, R, H);
    else af[B][R - FN] = Rows::frag(a, alane, R - FN, H);
  }
  template <int B, int H>
  __device__ __forceinline__ void read_all(const bf16* w, const bf16* a) {
    unrolled<0, FN + NA>([&](auto R) { read<B, decltype(R)::value, H>(w, a); });
  }
  // The products of register set B; between them the reads of half H (-1: none) of (w, a) into the other set,
  // and DEP calls of `dep`.  FRESH: the first of a tile, which add to nothing.
  template <int B, int H, int DEP, bool FRESH = false, class Dep>
  __device__ __forceinline__ void multiply(f32x4 (&acc)[FN][NA > 0 ? NA : 1], const bf16* w, const bf16* a, Dep dep) {
    if constexpr (NM == 0) {
      unrolled<0, DEP>([&](auto D) { dep(D); });
    } else {
      constexpr int NR = H >= 0 ? FN + NA : 0, PER = (2 * NR + NM - 1) / NM;  // reads behind an MFMA: in the first half
      unrolled<0, NM>([&](auto MC) {
        constexpr int m = decltype(MC)::value, j = m / NA, i = (j & 1) ? NA - 1 - m % NA : m % NA;
        acc[j][i] = mfma16(wf[B][j], af[B][i], FRESH ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[j][i]);
        unrolled<0, PER>([&](auto R) {
          constexpr int r = m * PER + decltype(R)::value;
          if constexpr (r < NR) read<B ^ 1, r, (H > 0 ? 1 : 0)>(w, a);
        });
        unrolled<0, DEP>([&](auto D) {
          constexpr int d = decltype(D)::value;
          if constexpr (((2 * d + 1) * NM) / (2 * DEP) == m) dep(D);
        });
        order_fence();
      });
    }
  }
};

constexpr int kStagingElems = 4096;  // a wave's share of the epilogue's staging

// Keeps `v` in its register from here on: the compiler waits for the load behind it now and not at
// its next use.
template <class T>
__device__ __forceinline__ void settle(T& v) {
  static_assert(sizeof(T) == 4, "one register");
  asm volatile("" : "+v"(v));
}

// Drives a workgroup through its (row tile, column block) pairs.  The tile program P supplies
//   P::G, P::Rows, P::Weights                  geometry and operands
//   P::Ids, P::Late                            per-tile values that come from loads; Late's depend on Ids'
//   gather(tile, ids) / late(tile, ids, late)  issue those loads
//   settle(ids) / settle(late)                 settle() each register of them
//   setup(tile, ids, A, W)                     operand set-up
//   epilogue(tile, acc, ids, late, staging)    acc [FN][fragment rows]; staging: kStagingElems of LDS per wave
//   EXCHANGE, finish(tile, staging)            if the waves leave values for each other there: behind a barrier
//   K, n_org[FN]                               contraction length, first columns of the fragments
// While tile t is multiplied, the ids of tile t+2, the late values of tile t+1 and the table entry of
// tile t+3 are on their way.  All of them settle at the end of tile t's epilogue: the compiler does
// not see the transfers, so its wait for any load is a wait for every transfer older than the
// youngest few, which cost a memory latency per tile in the middle of a stage; there the transfers
// have had the epilogue to arrive.
// The launch has `nb` column blocks; `first`: row tiles left out.
template <class P, class Args>
__device__ __forceinline__ void run_span_tiles(const Args& args, int nb, int max_tile_rows, int first = 0) {
  using G = typename P::G;
  using Sched = SpanSched<G>;
  Sched sched(args.table, nb, max_tile_rows, first);
  P prog(args);
  using Rows = typename P::Rows;
  using Weights = typename P::Weights;
  constexpr int FN = G::FN, AHEAD = G::AHEAD;
  constexpr int ROWS_AT = (AHEAD + 1) * Weights::ELEMS;  // the rows' ring lies behind the weights'
  static_assert((ROWS_AT + AHEAD * Rows::ELEMS) * sizeof(bf16) <= kSpanLds, "the rings fit the LDS");
  static_assert(Weights::ELEMS >= kSpanWaves * kStagingElems, "a stage of weights holds the epilogue's staging");
  bf16* const lds = dyn_lds();
  const uint32_t addr = lds_address(lds) + wave_id() * 1024;
  // slots by their byte offsets: of the stage before the one at hand, of that one, of the next one
  static_assert(AHEAD == 2, "three slots of weights, two of rows");
  constexpr uint32_t WSLOT = Weights::ELEMS * 2, ASLOT = Rows::ELEMS * 2;
  struct Ring {
    uint32_t wlast = 2 * WSLOT, w = 0, wnext = WSLOT, a = ROWS_AT * 2, anext = ROWS_AT * 2 + ASLOT;
    __device__ __forceinline__ void turn() {
      const uint32_t old = wlast, olda = a;
      wlast = w, w = wnext, wnext = old;
      a = anext, anext = olda;
    }
  } ring;
  auto at = [&](uint32_t offset) { return (const bf16*)((const char*)lds + offset); };

  TileCoord c0 = sched.next();
  if (!c0.valid) return;
  typename P::Ids g0, g1, g2;
  typename P::Late l0, l1;
  Rows A;
  Weights W;
  prog.gather(c0, g0);
  const SpanStages st(prog.K);
  prog.setup(c0, g0, A, W);
  int k = 0;  // k-origin of the stage to be requested
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
    const bf16 *wsrc = W.source(k), *asrc = A.source(k);
    unrolled<0, Weights::DEP>([&](auto D) { W.template deposit<decltype(D)::value>(wsrc, addr + s * WSLOT); });
    unrolled<0, Rows::DEP>([&](auto D) { A.template deposit<decltype(D)::value>(asrc, addr + ROWS_AT * 2 + s * ASLOT); });
    k = st.after(k);
  }
  TileCoord c1 = sched.next();
  g1 = g0;
  if (c1.valid) prog.gather(c1, g1);
  TileCoord c2 = sched.next();
  prog.settle(g0);
  prog.settle(g1);
  prog.late(c0, g0, l0);
  wait_vmcnt<(AHEAD - 1) * (Weights::DEP + Rows::DEP)>();
  __builtin_amdgcn_s_barrier();
  order_fence();
  g2 = g1;
  l1 = l0;
  while (true) {
    if (c2.valid) prog.gather(c2, g2);
    if (c1.valid) prog.late(c1, g1, l1);
    const typename Sched::Raw rn = sched.fetch();

    // this tile for a wave with NA fragment rows
    auto tile = [&](auto NAC) {
      constexpr int NA = decltype(NAC)::value;
      f32x4 acc[FN][NA > 0 ? NA : 1];
      SpanFrags<Rows, Weights, FN, NA> fr(c0.mbase, prog.n_org);
      // the next stage has landed, all but what was requested after it; every wave is done reading this one
      auto turn = [&] {
        wait_vmcnt<(AHEAD - 1) * Weights::DEP + (AHEAD - 2) * Rows::DEP>();
        wait_lgkm0();
        __builtin_amdgcn_s_barrier();
        order_fence();
      };
      fr.template read_all<0, 0>(at(ring.w), at(ring.a));
      order_fence();
      auto stage = [&](auto FRESH) {
        const bf16 *wsrc = W.source(k), *asrc = A.source(k);
        const uint32_t wto = addr + ring.wlast, ato = addr + ring.a;
        fr.template multiply<0, 1, Weights::DEP, decltype(FRESH)::value>(
            acc, at(ring.w), at(ring.a), [&](auto D) { W.template deposit<decltype(D)::value>(wsrc, wto); });
        turn();
        fr.template multiply<1, 0, Rows::DEP>(
            acc, at(ring.wnext), at(ring.anext), [&](auto D) { A.template deposit<decltype(D)::value>(asrc, ato); });
        k = st.after(k);
        ring.turn();
      };
      auto request_next_tile = [&] {
        k = 0;
        if (c1.valid) {
          prog.setup(c1, g1, A, W);
        } else {
          A.idle();
          W.idle();
        }
      };
      // The first stage by itself: its products start from zero, which a loop would have to write to 256 accumulation
      // registers before them.  In us, 8192 tokens, D = 2048, H = 1024, N = 128, K = 8: x.Wl1 466 -> 462, h.Wl2 270 -> 267,
      // recomputing GEMM 544 -> 541, dL/dx 451 -> 448, Wl1 gradient 634 -> 622, Wl2 gradient 330 -> 326.
      if (st.count == AHEAD) request_next_tile();
      stage(IntC<true>{});
      int t = 1, end = st.count == AHEAD ? st.count : st.count - AHEAD;
      while (true) {
        const int stop = min(end, st.full);
#pragma unroll 1
        for (; t < stop; ++t) stage(IntC<false>{});
        if (end == st.count) break;
        end = st.count;  // from here on the next tile's stages are requested
        request_next_tile();
      }
      if (st.tail) {
        const bf16 *wsrc = W.source(k), *asrc = A.source(k);
        unrolled<0, Weights::DEP>([&](auto D) { W.template deposit<decltype(D)::value>(wsrc, addr + ring.wlast); });
        fr.template read_all<0, 1>(at(ring.w), at(ring.a));
        fr.template multiply<0, -1, 0>(acc, at(ring.w), at(ring.a), [](auto) {});
        turn();
        unrolled<0, Rows::DEP>([&](auto D) { A.template deposit<decltype(D)::value>(asrc, addr + ring.a); });
        k = st.after(k);
        ring.turn();
      }
      // staging: where the finished tile's last weights were; every wave has read them, and the next ones are
      // requested behind the barrier below
      keep_in_place(acc);
      if constexpr (NA > 0) prog.epilogue(c0, acc, g0, l0, (bf16*)at(ring.wlast));
    };
    const int na = __builtin_amdgcn_readfirstlane(c0.na);
    if (na == 4) tile(IntC<8>{});
    else if (na == 3) tile(IntC<6>{});
    else if (na == 2) tile(IntC<4>{});
    else if (na == 1) tile(IntC<2>{});
    else tile(IntC<0>{});
    if constexpr (P::EXCHANGE) {
      wait_lgkm0();
      __builtin_amdgcn_s_barrier();
      prog.finish(c0, (bf16*)at(ring.wlast));
    }
    prog.settle(g2);
    prog.settle(l1);
    if (!c1.valid) break;
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    c0 = c1;
    c1 = c2;
    c2 = sched.resolve(rn);
    g0 = g1;
    g1 = g2;
    l0 = l1;
  }
  wait_vmcnt<0>();  // no transfer may outlive the workgroup's LDS
}

// Whether a launch over `cols` output columns takes these tiles rather than those of gemm_tile.hpp.  Not
// where most CUs would go without one (takes_narrow_tiles), nor with few rows per expert: a tile of few
// rows is a stream of weights, and then what is on the way counts, two to three stages of 32 k-values at
// any time in that ring, one of 64 here; nor in one round of one tile per expert with at most 512 k-values, where
// the start and the last stores are much of the time.  Otherwise by the rounds of tiles the CUs take, a tile costing 0.4
// for its weights and 0.6 for 256 rows, and of it all 0.8 here plus an epilogue that nothing hides,
// 0.07 of a contraction over 1024: an expert of 260 rows is two tiles here and one of 320 rows there.
// (The k-loop needs two stages.)
// Measured, there -> here in us (x.Wl1, h.Wl2, dL/dh, dL/dx): 8192 tokens, D = 2048, H = 1024, N = 128, K = 8
// 538 -> 498, 302 -> 286, 293 -> 252, 562 -> 493; 7680, D = 2176, H = 1152, N = 64, K = 6 438 -> 388, 257 -> 234,
// 260 -> 209, 459 -> 388; 4000, D = 1024, H = 512, N = 64, K = 4 (64 tiles of 320 rows, 81 of 256) 39 -> 47,
// 27 -> 31, 36 -> 27, 39 -> 43: here only dL/dh.  D = 512, H = 256, N = 96, 130
// rows per expert, x.Wl1 18.2 -> 20.8, dL/dx 18.2 -> 19.6: there.
// The routing is not known; the rows per expert are taken as those of one with the same chance for
// every expert, whose row counts spread by the root of their mean.  The choice is the wrong one for some loads without
// any spread: of 257 to 320 rows each, one tile of 320 would do where two are taken.  A choice that allowed for
// those would cost the others several times as much.  There -> here, 300 rows per expert, all the same | spread:
// x.Wl1 with D = 2048, H = 1024, N = 64 163 -> 178 | 218 -> 178, N = 128 327 -> 352 | 374 -> 355; h.Wl2 with N = 64 95 ->
// 101 | 116 -> 100; dL/dx 180 -> 186 | 221 -> 184.  A forward of such loads takes up to 9 % more than there, a step with its backward
// 0 to 6 % less.  (Tiles of six and four fragment rows instead of five and five, a wave row being two, changed
// nothing: 0.2 to 0.4 % more over 5760 launches.)
inline bool takes_span_tiles(int64_t msum, int64_t n, int64_t cols, int64_t contraction) {
  if (contraction < WideSpan::AHEAD * kSpan || takes_narrow_tiles(msum, n, cols) || few_rows_per_expert(msum, n)) return false;
  const double mean = (double)msum / n, spread = std::sqrt(mean), blocks = (double)cdiv64(cols, WideSpan::COLS);
  // row tiles per expert of at most `height` rows (normal spread, its tail by the logistic curve, which in
  // double precision is 1 from 24 spreads below the mean on)
  auto row_tiles = [&](double height) {
    double t = 1.0 + std::max(0.0, std::floor((mean - 24 * spread) / height));
    for (double k = t; k * height < mean + 6 * spread; ++k) t += 1.0 / (1.0 + std::exp(1.7 * (k * height - mean) / spread));
    return t;
  };
  auto tile_cost = [&](double tiles) { return 0.4 + 0.6 * mean / (tiles * StdTiles::MAX_ROWS); };
  const double tall = std::min(row_tiles(TallTiles::MAX_ROWS), row_tiles(StdTiles::MAX_ROWS)), ours = row_tiles(WideSpan::MAX_ROWS);
  if (contraction <= 512 && ours < 1.05 && n * blocks <= persistent_grid()) return false;
  const double rounds = n * ours * blocks / persistent_grid(), rest = rounds - std::floor(rounds);
  const double pieces = rest > 0.5 ? 1.0 : rest > 0.25 ? 0.65 : rest > 0.125 ? 0.45 : 0.3;  // SpanSched
  return (0.8 + 73.0 / contraction) * tile_cost(ours) * (std::floor(rounds) + pieces) <=
         tile_cost(tall) * std::ceil(n * tall * blocks / persistent_grid() - 0.05);
}

template <class Kernel, class Args>
inline int launch_span(Kernel kernel, const Args& a, LdsLimit& lim, hipStream_t st) {
  if (!allow_lds(kernel, kSpanLds, lim)) return MOMOE_ERR_LAUNCH;
  kernel<<<persistent_grid(), kSpanThreads, kSpanLds, st>>>(a);
  return launch_status();
}

// ---- ids ------------------------------------------------------------------------------------------
// Tokens of a tile's rows for SpanGatheredRows: lane l keeps that of row 32 * (l / 8) + 8 * wave + l % 8
struct FetchIds {
  int32_t tok;
  __device__ __forceinline__ void gather(const TileCoord& t, const int32_t* idx) {
    const int l = fresh_lane();
    tok = idx[t.row0 + min(32 * (l >> 3) + 8 * wave_id() + (l & 7), t.rows - 1)];
  }
  // of the row that lane l, this one, fetches in deposit j
  __device__ __forceinline__ int32_t of(int j, int l) const { return __shfl(tok, 8 * j + (l >> 3)); }
};

// Tokens of the 128 rows a wave holds in its accumulators: lane l keeps those of rows l and 64 + l
struct RowIds {
  int32_t tok[2];
  __device__ __forceinline__ void gather(const TileCoord& t, const int32_t* idx) {
    const int l = fresh_lane();
#pragma unroll
    for (int q = 0; q < 2; ++q) tok[q] = idx[t.row0 + min(t.mbase + 64 * q + l, t.rows - 1)];
  }
  __device__ __forceinline__ void settle() { momoe::settle(tok[0]), momoe::settle(tok[1]); }
};
// their gate weights
struct RowScales {
  float s[2];
  __device__ __forceinline__ void load(const TileCoord& t, const RowIds& g, const float* s_NM, int64_t ssn, int64_t ssm) {
#pragma unroll
    for (int q = 0; q < 2; ++q) s[q] = s_NM[(int64_t)t.expert * ssn + (int64_t)g.tok[q] * ssm];
  }
  __device__ __forceinline__ void settle() { momoe::settle(s[0]), momoe::settle(s[1]); }
  // of the row that lane l, this one, holds in fragment row i
  __device__ __forceinline__ float of(int i, int l) const { return __shfl(s[i / 4], 16 * (i % 4) + (l & 15)); }
};

// ---- coalesced epilogue stores ----------------------------------------------------------------------
// One 16-row fragment row of a wave at a time passes through a staging area (16 rows x WIDTH columns) and
// leaves as 16 bytes per lane, lanes along the rows: whole lines.  Wave-private: no barrier is
// involved.  With two areas in turn a row's reads travel while the one before it is stored.
template <int WIDTH>
struct SpanStager {
  static constexpr int CHUNKS = WIDTH / 8, PASSES = 16 * CHUNKS / 64;
  static constexpr int ELEMS = 16 * WIDTH;
  static_assert(2 * ELEMS <= kStagingElems, "two areas");
  static constexpr int ROWS_PER_BANK_ROW = 256 / (2 * WIDTH);
  static __device__ __forceinline__ int swz(int row) { return (row / ROWS_PER_BANK_ROW) & (CHUNKS - 1); }
  bf16* st;
  int l;  // fresh_lane() of the epilogue
  __device__ __forceinline__ SpanStager(bf16* staging, int lane) : st(staging + wave_id() * kStagingElems), l(lane) {}
  // this lane's four columns of fragment f
  __device__ __forceinline__ void put(int area, int f, bf16x4 v) const {
    const int row = l & 15;
    *(bf16x4*)(st + area * ELEMS + row * WIDTH + ((2 * f + (l >> 5)) ^ swz(row)) * 8 + ((l >> 4) & 1) * 4) = v;
  }
  // pass p: 8 columns from col(p) of row(p)
  __device__ __forceinline__ int row(int p) const { return p * (64 / CHUNKS) + l / CHUNKS; }
  __device__ __forceinline__ int col(int p) const { return ((l % CHUNKS) ^ swz(row(p))) * 8; }
  __device__ __forceinline__ bf16x8 get(int area, int p) const {
    return *(const bf16x8*)(st + area * ELEMS + row(p) * WIDTH + (l % CHUNKS) * 8);
  }
  // 8 rows, from 8 * (l / 16), of column 16 p + l % 16 of the 32 rows in areas `area` and `area` + 1
  __device__ __forceinline__ bf16x8 get_rows(int area, int p) const {
    const int row = 8 * (l >> 4) + ((l & 15) >> 2);  // (lds_read_tr4: this lane names the address of a neighbour's)
    auto at = [&](int r) {
      return st + (area + (r >> 4)) * ELEMS + (r & 15) * WIDTH + ((2 * p + ((l & 3) >> 1)) ^ swz(r & 15)) * 8 + (l & 1) * 4;
    };
    const bf16x4 lo = lds_read_tr4(at(row)), hi = lds_read_tr4(at(row + 4));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // as row(), col() and get() with a pass of 32 columns of 16 rows: 8 columns from 32 p + block_col() of block_row()
  __device__ __forceinline__ int block_row() const { return l >> 2; }
  __device__ __forceinline__ int block_col() const { return (l & 3) * 8; }
  __device__ __forceinline__ bf16x8 get_block(int area, int p) const {
    return *(const bf16x8*)(st + area * ELEMS + (l >> 2) * WIDTH + ((4 * p + (l & 3)) ^ swz(l >> 2)) * 8);
  }
};
__device__ __forceinline__ bf16x4 pack_bf16x4(f32x4 v, float s) {
  return bf16x4{(bf16)(v[0] * s), (bf16)(v[1] * s), (bf16)(v[2] * s), (bf16)(v[3] * s)};
}

// A wave's accumulators as `rows` rows, from row0, of a row-major matrix of `cols` columns, from column col0; scale(i) is that of
// the lane's row in fragment row i; lane = fresh_lane().  Rows behind the last one lie past a bound, a lane without columns
// names an offset past any.  (With a comparison and two selections for each store instead the vector unit, which all of this is
// bound by, had a ninth more to do: 8192 tokens, D = 2048, H = 1024, N = 128, K = 8, Wl1 gradient 648 -> 640 us, Wl2 gradient
// 332 -> 326, h.Wl2 270 -> 268, dL/dx 452 -> 449.  The epilogues of the SwiGLU products gain nothing from it: their bounds differ
// from store to store, and the scalar registers they take were spilled.)
template <bool STREAM = false, int FN, int NA, class Scale>
__device__ __forceinline__ void store_rows(f32x4 (&acc)[FN][NA], bf16* staging, bf16* out, int64_t row0, int rows, int cols,
                                           int col0, int lane, Scale scale) {
  using Stager = SpanStager<16 * FN>;
  const Stager stager(staging, lane);
  bf16* const first = out + row0 * cols + col0;  // uniform
  uint32_t off[Stager::PASSES];
#pragma unroll
  for (int p = 0; p < Stager::PASSES; ++p)
    off[p] = col0 + stager.col(p) < cols ? ((uint32_t)stager.row(p) * (uint32_t)cols + stager.col(p)) * 2 : 0xFFFFFFF0u;
  bf16x8 v[2][Stager::PASSES];
  auto store = [&](int i) {
    const uint32_t bytes = rows_of_fragment(16 * i, rows) * (uint32_t)cols * 2;
#pragma unroll
    for (int p = 0; p < Stager::PASSES; ++p)
      store16_below<STREAM>(first + (int64_t)(16 * i) * cols, off[p], bytes, v[i & 1][p]);
  };
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const float s = scale(i);
#pragma unroll
    for (int f = 0; f < FN; ++f) stager.put(i & 1, f, pack_bf16x4(acc[f][i], s));
    if (i > 0) store(i - 1);
#pragma unroll
    for (int p = 0; p < Stager::PASSES; ++p) v[i & 1][p] = stager.get(i & 1, p);
  }
  store(NA - 1);
}

}  // namespace momoe
