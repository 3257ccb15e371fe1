// Stages of the router's gate products: 64 k-values (rows) of 128 columns, k-strided, through registers into LDS.
#pragma once
#include "gemm_tile.hpp"

namespace momoe {

// A thread's pieces of a stage; what does not exist is zero.  Loads are unconditional, rows and columns clamped: under a
// branch each would be waited for before the next.
struct GateStage {
  static constexpr int THREADS = 256, ROWS = 64, COLS = 128;
  // elements of a row in LDS: the 4 rows of 16 lanes of a transposing read lie in different banks
  static constexpr int PITCH = COLS + 16, ELEMS = ROWS * PITCH;
  static constexpr int ACROSS = COLS / 8, STEP = THREADS / ACROSS, PIECES = ROWS / STEP;  // pieces of 16 bytes
  bf16x8 v[PIECES];
  // rows [row0, row0 + 64) of those below `end`, columns [0, cols) (a multiple of 8) from `base`, row pitch ld
  __device__ __forceinline__ void load(const bf16* base, int64_t ld, int cols, int row0, int end) {
    const int col = (threadIdx.x % ACROSS) * 8;
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      const int row = row0 + (int)threadIdx.x / ACROSS + q * STEP;
      const bf16x8 w = *(const bf16x8*)(base + (int64_t)min(row, end - 1) * ld + min(col, cols - 8));
      v[q] = row < end && col < cols ? w : bf16x8{};
    }
  }
  __device__ __forceinline__ void put(bf16* lds) const {
    const int col = (threadIdx.x % ACROSS) * 8;
#pragma unroll
    for (int q = 0; q < PIECES; ++q) *(bf16x8*)(lds + ((int)threadIdx.x / ACROSS + q * STEP) * PITCH + col) = v[q];
  }
  // 16 columns from `col` of k-values 32 h .. +31, as a fragment of v_mfma_f32_16x16x32_bf16
  static __device__ __forceinline__ bf16x8 frag(const bf16* lds, int col, int h) {
    const int l = threadIdx.x & 63;
    const bf16* p = lds + (32 * h + 8 * (l >> 4) + ((l & 15) >> 2)) * PITCH + col + 4 * (l & 3);
    const bf16x4 lo = lds_read_tr4(p), hi = lds_read_tr4(p + 4 * PITCH);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

}  // namespace momoe
