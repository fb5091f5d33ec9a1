// The f16 shared expert of long-run calls with enough of it (g5_linear's mx::matmul branch, glm5_kda.cpp:120;
// SwiGLU as in glm5_moe.cpp:66-74): two tiled f16 matrix products, gfx950.
//
//  k_shared_gemm<true>   gate and up of the same columns in one workgroup, SwiGLU at the end
//                        -> dsh_act (N, SI) f16
//  k_shared_gemm<false>  down -> dsh_dn as (N, H) f16, the linear's output, added by the combine
//
// Per output the arithmetic is dense_mfma's and its consumers': every k split accumulated
// from zero by 16x16x32 MFMAs in step order, the splits added in order.
//
// Bound by the LDS and L2 reads of the operands: at 500 rows of hidden 4096 and intermediate
// 1024 the two products are 12.6 GFLOP (10 us at 1.32 PFLOP/s) over 25 MB of weights. As
// tasks of 16 x 16 outputs and one k split each, inside the expert launches, every operand
// value was read from L2 once per 16 outputs and 32 bytes of partials written per output: the
// 500-row call went from 834 to 706 us, the 2048-row one from 1981 to 1327 (at 70 rows, on
// another card, 483 to 469).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "exl3_device.hpp"
#include "exl3_internal.hpp"
#include "moe_common.hpp"
#include "moe_dense.hpp"

namespace exl3d {

using exl3m::MoeArgs;

// Both operands are rows of consecutive k (token rows; output rows of the transposed
// weights), copied to LDS in parts of 64 k, 128 bytes per row unpadded, by the 16-byte
// direct-to-LDS load, 8 rows each: chunk c of row r at position c ^ (r / 2 % 8), so that
// the 16 rows of an MFMA operand read every bank once. Four part buffers (objects of their
// own, as the compiler tracks the copies per object), three of them in flight.
constexpr int kPartK = 64;
typedef __attribute__((address_space(3))) void gemm_lds_t;

__device__ __forceinline__ void gemm_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void gemm_copy(__amdgpu_buffer_rsrc_t src, uint32_t *dst, uint32_t vo) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (gemm_lds_t *)dst, 16, vo, 0, 0, 0);
}

// Workgroup: WR x WC waves; a wave has TM row tiles (16) and TN column tiles, for gate/up
// TN / 2 of each. kTile: rows of one LDS part, token rows first. (Two waves per SIMD: within
// 256 registers the sums of both levels stay out of the accumulation registers, which the
// additions cannot read.)
template <bool GU, int WR, int WC, int TM, int TN>
__global__ __launch_bounds__(64 * WR *WC) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_shared_gemm(MoeArgs a) {
  constexpr int kRows = 16 * TM * WR, kCols = 16 * TN * WC, kTile = kRows + kCols;
  constexpr int kWords = kTile * kPartK / 2;
  constexpr int kWaves = WR * WC, kCopies = kTile / 8 / kWaves;  // copies per wave and part
  __shared__ __align__(16) uint32_t b0[kWords], b1[kWords], b2[kWords], b3[kWords];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int in = GU ? a.H : a.SI;
  // output columns of the workgroup: kCols of H, or kCols / 2 of SI, gate's and up's
  const int n_cb = GU ? a.SI / (kCols / 2) : a.H / kCols;
  const int cb = blockIdx.x % n_cb;
  const int64_t row0 = (int64_t)(blockIdx.x / n_cb) * kRows;
  const int nr = (int)min<int64_t>(kRows, a.N - row0);
  const uint32_t row_bytes = 2u * in;
  const uint16_t *x = GU ? a.h : a.dsh_act;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(x + row0 * in), (short)0,
                                                                      (int)(nr * row_bytes), 0x00020000);
  // gate's and up's weights are one array, up's rows SI after gate's
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.sh_dense[GU ? 0 : 2], (short)0, (int)((uint32_t)(GU ? 2 * a.SI : a.H) * row_bytes), 0x00020000);
  // instruction i of a part copies tile rows 8i .. 8i + 7; this wave's are wave + kWaves j
  uint32_t vo[kCopies];
#pragma unroll
  for (int j = 0; j < kCopies; ++j) {
    const int r = 8 * (wave + kWaves * j) + (lane >> 3);  // tile row
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    int src = r;
    if (r >= kRows) {
      const int n = r - kRows;
      src = GU ? (n < kCols / 2 ? cb * (kCols / 2) + n : a.SI + cb * (kCols / 2) + n - kCols / 2) : cb * kCols + n;
    }
    vo[j] = (uint32_t)src * row_bytes + 16u * c;
  }
  const int n_parts = in / kPartK;
  auto issue = [&](int t, uint32_t *buf) {
    // (past the last part: that one again, never used)
    const uint32_t k = (uint32_t)min(t, n_parts - 1) * (2 * kPartK);
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
      static_assert(kRows % (8 * kWaves) == 0, "instruction j's rows are of one operand in every wave");
      gemm_copy(8 * kWaves * j < kRows ? rx : rw, buf + (wave + kWaves * j) * (8 * kPartK / 2), vo[j] + k);
    }
  };
  issue(0, b0);
  gemm_fence();
  issue(1, b1);
  gemm_fence();
  issue(2, b2);
  gemm_fence();
  const int l15 = lane & 15, g = lane >> 4, wr = wave % WR, wc = wave / WR;
  // operand chunk of 32-k step s: 4s + g, at row l15 of a tile (tiles start at multiples of 16
  // rows, so the swizzle is the lane's)
  int xo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) xo[s] = l15 * (kPartK / 2) + 4 * ((4 * s + g) ^ ((l15 >> 1) & 7));
  // first tile row of this wave's column tile n: gate's tiles, then up's
  auto col_row = [&](int n) {
    return kRows + (GU ? (n < TN / 2 ? 16 * (wc * (TN / 2) + n) : kCols / 2 + 16 * (wc * (TN / 2) + n - TN / 2))
                       : 16 * (wc * TN + n));
  };
  f32x4_ D[TM][TN], Y[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      D[m][n] = f32x4_{0.0f, 0.0f, 0.0f, 0.0f};
      Y[m][n] = f32x4_{-0.0f, -0.0f, -0.0f, -0.0f};  // -0 + v is v
    }
  const int split_parts = in / dense_mfma_splits(in) / kPartK;
  int ends = split_parts;
  // Part t in cur; its copies are this wave's oldest, two parts' copies were issued after
  // them. The wait (also for this wave's LDS reads) and the barrier: every wave's copies of
  // part t are in LDS and nobody reads the part before it, whose buffer takes part t + 3.
  auto run_part = [&](int t, uint32_t *cur, uint32_t *nxt) {
    constexpr int kLeft = 2 * kCopies;
    static_assert(kLeft < 64, "vmcnt field");
    gemm_fence();
    __builtin_amdgcn_s_waitcnt(0x0070 | (kLeft & 15) | ((kLeft >> 4) << 14));
    gemm_fence();
    __builtin_amdgcn_s_barrier();
    gemm_fence();
    issue(t + 3, nxt);
    gemm_fence();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f16x8_ A[TM], B[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m)
        A[m] = *reinterpret_cast<const f16x8_ *>(cur + xo[s] + 16 * (wr * TM + m) * (kPartK / 2));
#pragma unroll
      for (int n = 0; n < TN; ++n) B[n] = *reinterpret_cast<const f16x8_ *>(cur + xo[s] + col_row(n) * (kPartK / 2));
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) D[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[m], B[n], D[m][n], 0, 0, 0);
    }
    if (t + 1 == ends) {
      ends += split_parts;
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int n = 0; n < TN; ++n) {
#pragma unroll
          for (int i = 0; i < 4; ++i) Y[m][n][i] = Y[m][n][i] + D[m][n][i];
          D[m][n] = f32x4_{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
  };
  int t = 0;
  for (; t + 4 <= n_parts; t += 4) {
    run_part(t, b0, b3);
    run_part(t + 1, b1, b0);
    run_part(t + 2, b2, b1);
    run_part(t + 3, b3, b2);
  }
  if (n_parts % 4) {  // a multiple of 2: k is one of 128
    run_part(t, b0, b3);
    run_part(t + 1, b1, b0);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the copies past the last part
  const float L = rf16d(a.swiglu_limit);
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * (wr * TM + m) + 4 * g + i;
      if (r >= nr) continue;
      if constexpr (GU) {
#pragma unroll
        for (int n = 0; n < TN / 2; ++n)
          a.dsh_act[(row0 + r) * a.SI + cb * (kCols / 2) + 16 * (wc * (TN / 2) + n) + l15] =
              f32_to_f16(swiglu1(rf16d(Y[m][n][i]), rf16d(Y[m][n + TN / 2][i]), L));
      } else {
#pragma unroll
        for (int n = 0; n < TN; ++n)
          reinterpret_cast<uint16_t *>(a.dsh_dn)[(row0 + r) * a.H + cb * kCols + 16 * (wc * TN + n) + l15] =
              f32_to_f16(Y[m][n][i]);
      }
    }
}

template <bool GU, int WR, int WC, int TM, int TN>
static void shared_go(const MoeArgs &a, hipStream_t st) {
  constexpr int kRows = 16 * TM * WR, kCols = 16 * TN * WC;
  const int64_t tiles = (a.N + kRows - 1) / kRows;
  const int n_cb = GU ? a.SI / (kCols / 2) : a.H / kCols;
  k_shared_gemm<GU, WR, WC, TM, TN><<<(unsigned)(tiles * n_cb), 64 * WR * WC, 0, st>>>(a);
}

}  // namespace exl3d

namespace exl3h {

using exl3m::kLongRows;

// The f16 shared expert as wave tasks (dense_mfma: 16 rows x 16 outputs x one k split) beside
// the experts' workgroups, or as the two products, each a chain of k parts of its own, as long
// for a narrow intermediate. Tasks up to one set of resident waves (4 per SIMD), unless they
// push more than an eighth of a set of the gate/up launch's expert waves (their number at
// uniform routing) into a second round. What the shared expert adds to a call, us, tasks
// against products, by hidden, intermediate and rows:
//   2048, 128, 70 (1280 tasks) 2, 13       512, 128, 200 (1248) 5, 8     4096, 256, 70 (3840) 12, 21
//   2048, 384, 100 beside 64 experts of 512 (2688 gate/up tasks, 2028 expert waves) 18, 14
//   3072, 128, 100 beside 160 of 384 (896, 3530) 6, 18
//   1024, 256, 200 (4992) 14, 11           2048, 256, 130 (4608) 20, 12  (8-wave workgroups)
constexpr int64_t kResidentWaves = 4096;

bool shared_products(int64_t N, int H, int SI, int I, int E, int topk) {
  const int64_t gu = 2 * exl3d::dense_mfma_tasks(N, H, SI);
  if (gu + exl3d::dense_mfma_tasks(N, SI, H) > kResidentWaves) return true;
  const double distinct = E * (1.0 - std::pow(1.0 - (double)topk / E, (double)N));
  const double experts = std::max(distinct, (double)N * topk / kLongRows) * 2 * (I / 32);
  return experts <= kResidentWaves && experts + gu > kResidentWaves + kResidentWaves / 8;
}

// 128 x 128 tiles (8 waves, one workgroup per CU) or 64 x 64 ones (4 waves, two per CU), for each
// product by its rounds of workgroups: a round of big tiles takes about 1.5 of small ones.
// Both products with the rest of a small layer, us, small against big tiles, by hidden and
// intermediate: 4096, 128 at 1024 rows 137, 152 and at 2048 180, 191; 512, 1024 at 1024 65, 72;
// 2048, 1024 at 1100 121, 116; 4096, 1024 at 2048 234, 222; 4096, 2048 at 1000 197, 181.
static bool big_tiles(int64_t rows, int64_t cols) {
  const int64_t big = (rows + 127) / 128 * (cols / 128), small = (rows + 63) / 64 * (cols / 64);
  return 3 * ((big + 255) / 256) < 2 * ((small + 511) / 512);
}

exl3_status launch_shared_dense(exl3m::MoeArgs a, hipStream_t st) {
  if (reinterpret_cast<uintptr_t>(a.h) % 4) {
    // the direct-to-LDS loads want dwords: rows at an odd f16 go through the shared slots of
    // xrot, which only a trellis shared expert uses
    uint16_t *x = a.xrot + (int64_t)a.P * 2 * a.H;
    EXL3_HIP(hipMemcpyAsync(x, a.h, (size_t)a.N * a.H * 2, hipMemcpyDeviceToDevice, st));
    a.h = x;
  }
  if (big_tiles(a.N, 2 * (int64_t)a.SI)) exl3d::shared_go<true, 4, 2, 2, 4>(a, st);
  else exl3d::shared_go<true, 2, 2, 2, 2>(a, st);
  if (big_tiles(a.N, a.H)) exl3d::shared_go<false, 4, 2, 2, 4>(a, st);
  else exl3d::shared_go<false, 2, 2, 2, 2>(a, st);
  EXL3_LAUNCHED("k_shared_gemm");
  return EXL3_OK;
}

}  // namespace exl3h
