// The trellis linear of many token rows: a workgroup computes 16 * RB rows x 32 columns per
// wave over the whole k range, each wave step's weights decoded once for all RB row blocks,
// and ends with the output Hadamard (or the raw f32 rows). Rows arrive rotated and in the
// staged k order (k_stage_rows). Instantiated in qmv_rows_k*.hip.
//
// Per output the arithmetic is k_qmv's and k_qmv_finalize's: every k slice accumulated from
// zero in step order by the same MFMAs, the slices' sums added in slice order, then the
// output Hadamard; so a row has the same bits as in a call of its own.
//
// Bound by the matrix cores with the decode beside them: 1000 rows x 8192 x 4096 are 67
// GFLOP, 51 us at the 1.32 PFLOP/s of a large library f16 product, and the decode (3.5 to 4.1
// VALU instructions per weight) runs once per 128 rows.
#pragma once

#include <type_traits>
#include <utility>

#include "exl3_device.hpp"
#include "exl3_internal.hpp"
#include "qmv_core.hpp"
#include "rows_lds.hpp"

namespace exl3d {

// One of the two part buffers (objects of their own, so that reads of one are not held back
// for the copies into the other); at the end it holds the f32 sums of 8 RB rows x 128 columns.
template <int RB>
constexpr int kRowsBufWords = 16 * RB * 4 * kRowsChunks;

struct RowsArgs {
  const uint16_t *xrot;  // (members, rows, in) f16, staged k order
  int64_t rows;
  int in, out;
  int row_tiles, col_groups, members;
  float *y32;            // (members, rows, out) raw sums, or
  uint16_t *y16;         // (members, rows, out) through the output Hadamard
  exl3h::PtrTable trellis, svh;
};

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>)
template <int... I, typename F>
__device__ __forceinline__ void rows_each(std::integer_sequence<int, I...>, F &&f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Position of column c of row r in the f32 tile (128 words a row): the four row groups of an
// accumulator land on different banks.
__device__ __forceinline__ int rows_col(int r, int c) { return c ^ (((r >> 2) & 1) << 5) ^ (((r >> 3) & 1) << 3); }

// (Waves per SIMD: the 64-row tile of K <= 4 fits 168 registers. At K = 5 it spilled 16 to 41
// of them under that bound: 4096 x 24576 at 17 rows took 48.7, 45.2 and 40.6 us by codebook,
// without spills 42.8, 42.1 and 38.5; the slice path 46.5, 45.8 and 45.9.)
template <int K, int CB, int RB, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(RB > 4 || K > 4 ? 2 : 3))) void k_qmv_rows(RowsArgs a) {
  static_assert(!dup_cb(CB), "reference-form weights");
  constexpr int PD = 2;
  __shared__ __align__(16) uint32_t buf_a[kRowsBufWords<RB>], buf_b[kRowsBufWords<RB>];
  __shared__ u32x4 slots[WAVES][slot_chunks(K)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // work items go to the 8 XCDs in contiguous ranges, row tiles fastest: the row tiles of one
  // column group read its weights through one L2, so they come from HBM once
  const int T = a.row_tiles * a.col_groups * a.members;
  const int x = blockIdx.x & 7, q = T >> 3, rem = T & 7;
  const int item = x * q + min(x, rem) + ((int)blockIdx.x >> 3);
  const int rt = item % a.row_tiles, cg = (item / a.row_tiles) % a.col_groups, member = item / a.row_tiles / a.col_groups;
  const int np = cg * WAVES + wave;
  const bool active = np < a.out / 32;
  const int64_t row0 = (int64_t)rt * (16 * RB);
  const int nr = (int)min<int64_t>(16 * RB, a.rows - row0);
  const int k_tiles = a.in / 16, total = k_tiles / kStepTiles, n_parts = total / kRowsPart;
  const int slice_parts = slice_steps(k_tiles) / kRowsPart;
  const uint32_t row_bytes = 2u * a.in;
  const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.xrot + ((int64_t)member * a.rows + row0) * a.in), (short)0, (int)(nr * row_bytes), 0x00020000);
  u32x4 *slot = slots[wave];

  const StepLane sl = step_lane();
  const int wbase = (sl.kt * 2 + sl.nt) * 8 * K;
  // A operand (step s of the part, half jp) of this lane's row: chunk 8s + 2kt + jp
  int xo[kRowsPart][2];
#pragma unroll
  for (int s = 0; s < kRowsPart; ++s)
#pragma unroll
    for (int jp = 0; jp < 2; ++jp)
      xo[s][jp] = (lane & 15) * (4 * kRowsChunks) + 4 * ((8 * s + 2 * sl.kt + jp) ^ (lane & 15));
  // An idle wave (past the last column) runs along on n-pair 0 and stores nothing.
  SliceStream<K, PD> S;
  const uint32_t vo = rows_voff<WAVES>(row_bytes, wave);
  rows_issue<RB, WAVES>(src, vo, row_bytes, 0, wave, buf_a);
  rows_fence();
  S.start((const uint32_t *)a.trellis.p[member], k_tiles, a.out / 16, 0, active ? np : 0);
  // sums of the current slice and of the ones before it (-0 + v is v, a zero's sign included)
  f32x4 D[RB][2], Y[RB][2];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    D[r][0] = D[r][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    Y[r][0] = Y[r][1] = f32x4{-0.0f, -0.0f, -0.0f, -0.0f};
  }
  // Waits for this wave's copies of a part: the ring loads of the PD steps issued after them
  // may stay in flight (loads complete in issue order; the fences keep the copies and the
  // ring loads in the order written). The barrier then makes every wave's copies visible; it
  // carries no __syncthreads fences, which would wait for every load.
  constexpr int kInFlight = PD * (K > 4 ? 2 : 1);
  auto copies_done = [&] {
    rows_fence();
    __builtin_amdgcn_s_waitcnt(0x0F70 | kInFlight);
    rows_fence();
    __builtin_amdgcn_s_barrier();
    rows_fence();
  };
  constexpr int kG = RB / 4, kGroups = kRowsPart * 2 * kG;  // groups of 4 row blocks, per half step
  static_assert(kGroups % 2 == 0, "operand registers alternate");
  f16x8 A[2][4];
  auto read_group = [&](int g, const uint32_t *buf) {
    const int s = g / (2 * kG), h = g / kG % 2, r0 = 4 * (g % kG);
#pragma unroll
    for (int r = 0; r < 4; ++r) A[g & 1][r] = lds_a(buf + xo[s][h] + (r0 + r) * (16 * 4 * kRowsChunks));
  };
  auto load_step = [&](int step, StepLoads<K> &L) {  // (past the last step: that one again)
    step_load<K>(S.rsrc, S.vo0, S.vo1, S.so0 + (uint32_t)min(step, total - 1) * S.step_bytes, L);
  };
  copies_done();
  rows_issue<RB, WAVES>(src, vo, row_bytes, 16 * kRowsChunks, wave, buf_b);
  rows_fence();
  uint32_t W[2][K + 1];  // ring words of this step and the next
  f16x8 B[2][2];         // operands of this half step and the next
  step_words<K>(slot, wbase, sl.m, S.L[0], W[0]);
  load_step(PD, S.L[0]);
  {
    uint32_t F[K + 1];
    lane_funnels<K>(W[0], F);
    B[0][0] = b_packed<K, CB, 0>(W[0], F);
    B[0][1] = b_packed<K, CB, 4>(W[0], F);
  }
  read_group(0, buf_a);
  // Part t, its rows in cur, the next part's in nxt (copied while this one is computed).
  // Software pipeline: a group's operands are read from LDS during the group before it, a
  // half step's weights decoded during the half step before it (the pin below keeps the
  // compiler from sinking a part's last decode past the branch at its end), and the barrier
  // of the next part is met before the last group's MFMAs.
  auto run_part = [&](int t, uint32_t *cur, uint32_t *nxt) {
    rows_each(std::make_integer_sequence<int, kRowsPart * 2>{}, [&](auto half) {
      constexpr int s = decltype(half)::value / 2, h = decltype(half)::value % 2;
      uint32_t F[K + 1];
      if constexpr (h == 0) {
        step_words<K>(slot, wbase, sl.m, S.L[(s + 1) & 1], W[(s + 1) & 1]);
        load_step(t * kRowsPart + s + 1 + PD, S.L[(s + 1) & 1]);
        lane_funnels<K>(W[s & 1], F);
      } else {
        lane_funnels<K>(W[(s + 1) & 1], F);
      }
      rows_each(std::make_integer_sequence<int, kG>{}, [&](auto grp) {
        constexpr int gg = decltype(grp)::value, g = decltype(half)::value * kG + gg;
        constexpr bool last = g + 1 == kGroups;
        if constexpr (last) {
          // every ring load of this part is issued; this wave's reads of cur are done once
          // the last operands are in, so other waves' copies may land there after the barrier
          asm volatile("" : "+v"(A[g & 1][0]), "+v"(A[g & 1][1]), "+v"(A[g & 1][2]), "+v"(A[g & 1][3]));
          copies_done();
          // (past the last part: bytes that are never used)
          rows_issue<RB, WAVES>(src, vo, row_bytes, (uint32_t)(t + 2) * (16 * kRowsChunks), wave, cur);
          rows_fence();
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          constexpr int gn = (g + 1) % kGroups, sn = gn / (2 * kG), hn = gn / kG % 2;
          A[(g + 1) & 1][r] = lds_a((last ? nxt : cur) + xo[sn][hn] + (4 * (gn % kG) + r) * (16 * 4 * kRowsChunks));
        }
        if constexpr (gg == 0) {
          constexpr int hn = h == 0 ? 1 : 0;
          B[1 - h][0] = b_packed<K, CB, 16 * hn>(W[(s + 1 - hn) & 1], F);
          B[1 - h][1] = b_packed<K, CB, 16 * hn + 4>(W[(s + 1 - hn) & 1], F);
          asm volatile("" : "+v"(B[1 - h][0]), "+v"(B[1 - h][1]));
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          D[4 * gg + r][0] = mfma16(A[g & 1][r], B[h][0], D[4 * gg + r][0]);
          D[4 * gg + r][1] = mfma16(A[g & 1][r], B[h][1], D[4 * gg + r][1]);
        }
      });
    });
  };
  // the slices' sums in slice order
  int ends = slice_parts;
  auto end_part = [&](int t) {
    if (t + 1 != ends) return;
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 4; ++i) Y[r][h][i] = Y[r][h][i] + D[r][h][i];
        D[r][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
    ends += slice_parts;
  };
  for (int t = 0; t + 2 <= n_parts; t += 2) {
    run_part(t, buf_a, buf_b);
    end_part(t);
    run_part(t + 1, buf_b, buf_a);
    end_part(t + 1);
  }
  if (n_parts & 1) {
    run_part(n_parts - 1, buf_a, buf_b);
    end_part(n_parts - 1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the copies past the last part

  // The sums through LDS, 128 columns (4 waves) at a time: the first half of the tile's
  // rows in one buffer, the rest in the other; then a wave per row.
  float *f_a = reinterpret_cast<float *>(buf_a), *f_b = reinterpret_cast<float *>(buf_b);
  for (int w0 = 0; w0 < WAVES; w0 += 4) {
    const int col0 = (cg * WAVES + w0) * 32;
    if (col0 >= a.out) break;  // the same for every wave
    __syncthreads();
    if (active && wave >= w0 && wave < w0 + 4) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rr = 16 * (r % (RB / 2)) + d_row(i);
          float *f = (r < RB / 2 ? f_a : f_b) + rr * 128;
          f[rows_col(rr, (wave - w0) * 32 + d_col(0))] = Y[r][0][i];
          f[rows_col(rr, (wave - w0) * 32 + d_col(1))] = Y[r][1][i];
        }
    }
    __syncthreads();
    float s0 = 0.0f, s1 = 0.0f;
    if (!a.y32) {
      const uint32_t sv = *reinterpret_cast<const uint32_t *>((const uint16_t *)a.svh.p[member] + col0 + 2 * lane);
      s0 = f16_to_f32((uint16_t)(sv & 0xffffu));
      s1 = f16_to_f32((uint16_t)(sv >> 16));
    }
    constexpr int kB = 4;  // rows per wave at a time
    for (int rb = kB * wave; rb < nr; rb += kB * WAVES) {
      float v0[kB], v1[kB];
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        const int r = rb + j;
        const float2 v = *reinterpret_cast<const float2 *>((r < 8 * RB ? f_a : f_b) + r % (8 * RB) * 128 +
                                                           rows_col(r, 2 * lane));
        v0[j] = v.x;
        v1[j] = v.y;
      }
      const int64_t o = ((int64_t)member * a.rows + row0 + rb) * a.out + col0 + 2 * lane;
      if (a.y32) {
#pragma unroll
        for (int j = 0; j < kB; ++j)
          if (rb + j < nr) *reinterpret_cast<float2 *>(a.y32 + o + (int64_t)j * a.out) = make_float2(v0[j], v1[j]);
      } else {
        const float t0[kB] = {s0, s0, s0, s0}, t1[kB] = {s1, s1, s1, s1};
        wave_had_post_n<kB>(v0, v1, t0, t1);
#pragma unroll
        for (int j = 0; j < kB; ++j)
          if (rb + j < nr) *reinterpret_cast<uint32_t *>(a.y16 + o + (int64_t)j * a.out) = pack_f16x2(v0[j], v1[j]);
      }
    }
  }
}

}  // namespace exl3d

namespace exl3h {

template <int K, int CB>
static void qmv_rows_go(int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st) {
  const unsigned grid = (unsigned)(a.row_tiles * a.col_groups * a.members);
  if (rb == 8 && waves == 8) exl3d::k_qmv_rows<K, CB, 8, 8><<<grid, 512, 0, st>>>(a);
  else if (rb == 8) exl3d::k_qmv_rows<K, CB, 8, 4><<<grid, 256, 0, st>>>(a);
  else exl3d::k_qmv_rows<K, CB, 4, 4><<<grid, 256, 0, st>>>(a);
}

template <int K>
static void qmv_rows_cb(int cb, int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st) {
  switch (cb) {
    case 0: qmv_rows_go<K, 0>(rb, waves, a, st); break;
    case 1: qmv_rows_go<K, 1>(rb, waves, a, st); break;
    default: qmv_rows_go<K, 2>(rb, waves, a, st);
  }
}

// Row blocks rb (8 or 4) and waves (8 or 4; 4 for rb = 4) per workgroup; defined in
// qmv_rows_k14.hip and qmv_rows_k58.hip.
void launch_qmv_rows_k14(int K, int cb, int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st);
void launch_qmv_rows_k58(int K, int cb, int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st);

}  // namespace exl3h
