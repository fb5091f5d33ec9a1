// Activation rows in the staged k order (qmv_core.hpp), copied from memory to LDS part by
// part by the direct-to-LDS loads, for the kernels that decode a weight once for many rows.
#pragma once

#include <hip/hip_runtime.h>

#include "qmv_core.hpp"

namespace exl3d {

// Rows are copied to LDS in parts of 2 wave steps (a slice is 2, 4 or 8), double-buffered:
// 256 bytes per row, unpadded, the 16-byte chunk c of row r at position c ^ (r % 16). A lane
// of the 16-byte direct-to-LDS load lands at the next 16 bytes, so one load takes 4 rows,
// and the 16 rows of an A operand read 16 different chunk positions (no bank conflicts).
constexpr int kRowsPart = 2;                                   // wave steps per part
constexpr int kRowsChunks = kRowsPart * kStepTiles * 8 / 4;    // 16-byte chunks of a row's part
static_assert(kRowsChunks == 16, "one chunk position per row of an A operand");
typedef __attribute__((address_space(3))) void rows_lds_t;

// This wave's share of a part's rows: instruction i copies rows 4i .. 4i + 3 (rows past the
// resource are zeros, not skipped, so that every wave issues the same number and the compiler
// can count them). vo: the lane's offset of instruction `wave` at the row's start
// (rows_voff); the lane's chunk position is the same in all of a wave's instructions, whose
// rows are 4 WAVES apart.
template <int WAVES>
__device__ __forceinline__ uint32_t rows_voff(uint32_t row_bytes, int wave) {
  static_assert(WAVES % 4 == 0, "rows 16n apart keep their chunk positions");
  const uint32_t lane = threadIdx.x & 63, r = 4 * wave + (lane >> 4);
  return r * row_bytes + 16u * ((lane & 15) ^ (r & 15));
}
template <int RB, int WAVES>
__device__ __forceinline__ void rows_issue(__amdgpu_buffer_rsrc_t src, uint32_t vo, uint32_t row_bytes,
                                           uint32_t kbyte0, int wave, uint32_t *buf) {
#pragma unroll
  for (int j = 0; j < 4 * RB / WAVES; ++j)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (rows_lds_t *)(buf + (wave + j * WAVES) * (16 * kRowsChunks)), 16,
                                             vo + (kbyte0 + j * (4 * WAVES) * row_bytes), 0, 0, 0);
}

// Keeps memory operations (the copies, the ring loads) in the order written.
__device__ __forceinline__ void rows_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace exl3d
