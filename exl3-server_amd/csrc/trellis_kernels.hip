// Trellis tensor kernels for gfx950: decode (W_hat), reconstruct (W), the Hadamard
// steps, and the dequant-GEMV (QMV) with its split-sum / output-Hadamard epilogue.
//
// Reference counterparts (muyouming/exl3-server):
//   decode       exl3.cpp:101-125      (bit-exact)
//   reconstruct  exl3.cpp:152-209      (bit-exact: same f32 butterfly order, one RNE)
//   hadamard     trellis_gemm.cpp:367-400, 582-603 (same rounding points)
//   qmv          trellis_gemm.cpp:30-141 (Metal scalar QMV) + mx::sum over splits
//                (:980, :1185) + the output Hadamard (:1186)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <utility>

#include "exl3_device.hpp"
#include "exl3_internal.hpp"
#include "qmv_core.hpp"
#include "qmv_rows.hpp"

using namespace exl3d;

namespace {

// ---------------------------------------------------------------------------------
// decode: one workgroup per tile, one thread per stream position.
// ---------------------------------------------------------------------------------
__device__ __forceinline__ int tile_element(int p) {
  const int L = p >> 3, i = p & 7, q = i & 3;
  const int row = 2 * (L & 3) + (q < 2 ? q : q + 6);
  const int col = (L >> 2) + 8 * (i >> 2);
  return row * 16 + col;
}

__device__ __forceinline__ uint32_t tile_state_rt(const uint32_t *__restrict__ tile, int K, int p) {
  const int nw = 8 * K;
  const int lb = (p + 1) * K - 1;  // ring bit of the state's LSB
  const int last = lb >> 5;
  const uint32_t lo = tile[last % nw];
  const uint32_t hi = tile[(last - 1 + nw) % nw];
  const uint64_t pair = ((uint64_t)hi << 32) | lo;
  return (uint32_t)(pair >> (31 - (lb & 31))) & 0xffffu;
}

template <int CB>
__global__ __launch_bounds__(256) void k_decode(const uint32_t *__restrict__ trellis, int K,
                                                int tiles_n, int out, uint16_t *__restrict__ w_hat) {
  const int tn = blockIdx.x, tk = blockIdx.y, p = threadIdx.x;
  const uint32_t *tile = trellis + ((int64_t)tk * tiles_n + tn) * 8 * K;
  const f16 v = decode_one<CB>(tile_state_rt(tile, K, p));
  const int e = tile_element(p);
  w_hat[(int64_t)(tk * 16 + (e >> 4)) * out + tn * 16 + (e & 15)] = bitcast<uint16_t>(v);
}

// ---------------------------------------------------------------------------------
// reconstruct: one workgroup of 4 waves per 128x128 block, the operation order of
// exl3.cpp:156-197 element for element: the left butterflies (across rows), the row scale,
// the right butterflies (across columns), the column scale and one RNE.
//
// Bound by VALU issue beside the memory floor (about 8,500 wave instructions per block; 4096 x
// 4096 K4: 16 us of issue, 42 MB or 8.2 us at 5.1 TB/s). The rows' butterflies stay in
// registers: a thread decodes 2 columns x 32 rows straight from its ring words, the stages of
// 1 to 16 rows are its own, those of 32 and 64 rows exchange lanes 16 and 32 apart. The block
// then goes through LDS 64 rows at a time (32 KB, so 4 workgroups share a CU) to a wave per
// row for the column stages and whole-row stores. Measured at that shape: 20 us, where
// 14 barriered passes over the block in 66 KB of LDS took 121.
// ---------------------------------------------------------------------------------
// v[i] <- the butterfly of v[i] and the value of the lane D (16 or 32) away.
template <int D, int N>
__device__ __forceinline__ void lane_butterfly(float (&v)[N]) {
  const float sgn = (threadIdx.x & D) ? -1.0f : 1.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    // r0 = the lower lane's value, r1 = the upper lane's, in both lanes
    const int x = __builtin_bit_cast(int, v[i]);
    const auto r = D == 32 ? __builtin_amdgcn_permlane32_swap(x, x, false, false)
                           : __builtin_amdgcn_permlane16_swap(x, x, false, false);
    v[i] = __builtin_fmaf(sgn, __builtin_bit_cast(float, (int)r[1]), __builtin_bit_cast(float, (int)r[0]));
  }
}

template <int K, int CB, int T>
__device__ __forceinline__ void decode_column_pair(const uint32_t (&W)[K + 1], const uint32_t (&F)[K + 1],
                                                   float (&v)[2][32], int j) {
  // stream position T of the lane's 32: k-row 2 (T / 8) + {0, 1, 8, 9}[T % 4], column half T / 4 % 2
  constexpr int row = 2 * (T / 8) + (T % 4 < 2 ? T % 4 : T % 4 + 6);
  v[T / 4 % 2][16 * j + row] = (float)decode_one<CB>(lane_state<K, T>(W, F));
}
template <int K, int CB, int... T>
__device__ __forceinline__ void decode_columns(const uint32_t (&W)[K + 1], const uint32_t (&F)[K + 1],
                                               float (&v)[2][32], int j, std::integer_sequence<int, T...>) {
  (decode_column_pair<K, CB, T>(W, F, v, j), ...);
}

template <int K, int CB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_reconstruct(
    const uint32_t *__restrict__ trellis, int tiles_n, int out, const uint16_t *__restrict__ suh,
    const uint16_t *__restrict__ svh, uint16_t *__restrict__ w) {
  __shared__ __align__(16) float buf[64 * 128];
  const int cbk = blockIdx.x, rbk = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // lane: columns m and m + 8 of tile column 2 wave + lane / 8 % 2, rows 32 q .. 32 q + 31
  const int m = lane & 7, tc = 2 * wave + ((lane >> 3) & 1), q = lane >> 4;
  uint32_t W[2][K + 1];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t *tile = trellis + ((int64_t)(rbk * 8 + 2 * q + j) * tiles_n + cbk * 8 + tc) * 8 * K;
    W[j][0] = tile[(m * K + 8 * K - 1) % (8 * K)];
#pragma unroll
    for (int i = 0; i < K; ++i) W[j][i + 1] = tile[m * K + i];
  }
  float v[2][32];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    uint32_t F[K + 1];
    lane_funnels<K>(W[j], F);
    decode_columns<K, CB>(W[j], F, v, j, std::make_integer_sequence<int, 32>{});
  }
#pragma unroll
  for (int len = 1; len < 32; len <<= 1)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 32; ++i)
        if (!(i & len)) {
          const float a = v[h][i], b = v[h][i + len];
          v[h][i] = a + b;
          v[h][i + len] = a - b;
        }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    lane_butterfly<16>(v[h]);
    lane_butterfly<32>(v[h]);
  }
  const uint16_t *su = suh + rbk * 128 + 32 * q;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const float s = f16_to_f32(su[i]) * kHadScale;
    v[0][i] = v[0][i] * s;
    v[1][i] = v[1][i] * s;
  }
  const uint16_t *sv = svh + cbk * 128 + 2 * lane;
  const float t0 = f16_to_f32(sv[0]) * kHadScale, t1 = f16_to_f32(sv[1]) * kHadScale;
  // 64 rows at a time; column c of a row whose bit 5 is set at c ^ 32, so that the two row
  // quarters that write together fall on different banks
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    if (p) __syncthreads();  // the first half has been read
    if ((q >> 1) == p) {
      float *b = buf + (q & 1) * 32 * 128 + ((tc * 16 + m) ^ ((q & 1) * 32));
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        b[i * 128] = v[0][i];
        b[i * 128 + 8] = v[1][i];  // (the swizzle leaves bit 3 alone)
      }
    }
    __syncthreads();
    constexpr int kB = 8;  // rows per wave at a time
#pragma unroll 1
    for (int r0 = kB * wave; r0 < 64; r0 += 4 * kB) {
      float x0[kB], x1[kB];
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const float2 x = *reinterpret_cast<const float2 *>(buf + (r0 + i) * 128 + ((2 * lane) ^ (r0 & 32)));
        x0[i] = x.x;
        x1[i] = x.y;
      }
      wave_fwht128_n<kB>(x0, x1);
      uint16_t *o = w + (int64_t)(rbk * 128 + 64 * p + r0) * out + cbk * 128 + 2 * lane;
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const uint32_t y = pack_f16x2(x0[i] * t0, x1[i] * t1);
        __builtin_memcpy(o + (int64_t)i * out, &y, 4);
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// Hadamard pre/post: one wave per (row, 128-block).
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_hadamard(const uint16_t *__restrict__ x16,
                                                  const float *__restrict__ x32, int64_t rows,
                                                  int n, exl3h::PtrTable s,
                                                  int64_t rows_per_member,
                                                  uint16_t *__restrict__ y) {
  const int lane = threadIdx.x & 63;
  const int64_t gw = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int nb = n / 128;
  if (gw >= rows * nb) return;
  const int blk = (int)(gw % nb);
  const int64_t row = gw / nb;
  const uint16_t *sv = (const uint16_t *)s.p[row / rows_per_member] + blk * 128 + 2 * lane;
  const int64_t o = row * n + blk * 128 + 2 * lane;
  float v0, v1;
  if (x16) {
    v0 = f16_to_f32(x16[o]);
    v1 = f16_to_f32(x16[o + 1]);
    wave_had_pre(v0, v1, f16_to_f32(sv[0]), f16_to_f32(sv[1]));
  } else {
    v0 = x32[o];
    v1 = x32[o + 1];
    wave_had_post(v0, v1, f16_to_f32(sv[0]), f16_to_f32(sv[1]));
  }
  y[o] = f32_to_f16(v0);
  y[o + 1] = f32_to_f16(v1);
}

// ---------------------------------------------------------------------------------
// QMV: grid (groups of column blocks, k-slices x row passes, members); 4 waves per
// workgroup, wave w owns n-pair 4*cb + w of each 128-column block cb of its group. The
// workgroup stages its slice of up to 16 xhat rows into LDS in the MFMA k order and writes
// the slice partials part[member][slice][row][col].
// ---------------------------------------------------------------------------------
// Bound by decode VALU, the rotation of the rows beside it: a workgroup rotates its slice of
// every row whatever its columns, so a group of blocks (kGroup) rotates once for all of them
// and keeps one ring-word stream over them (waves per SIMD as in the expert kernels).
// The slice partials of an n-pair's rows below nr, from p (its first row and column).
__device__ __forceinline__ void qmv_store(float *p, int out, int nr, const f32x4 &D0, const f32x4 &D1) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = d_row(i);
    if (r < nr) {
      p[(int64_t)r * out + d_col(0)] = D0[i];
      p[(int64_t)r * out + d_col(1)] = D1[i];
    }
  }
}

template <int K, int CB, int PD, bool kGroup>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kGroup ? (K <= 4 ? 7 : 6) : 1))) void k_qmv(exl3h::PtrTable trellis, int tiles_n, int in,
                                             int out, const uint16_t *__restrict__ xhat,
                                             int64_t x_member_stride, int64_t rows,
                                             int pass_rows, float *__restrict__ part,
                                             exl3h::PtrTable suh, int rotate, int group) {
  constexpr bool kDup = dup_cb(CB);
  // one ring-word slot per wave, then the slice's staged rows (pass_rows of them: the
  // launch sizes the LDS to the pass, so a one-row call is not held to the occupancy of
  // a 16-row one)
  extern __shared__ u32x4 qmv_smem[];
  u32x4 *slots = qmv_smem;
  uint32_t *xs = reinterpret_cast<uint32_t *>(qmv_smem + 4 * slot_chunks(K));
  const int k_tiles = in / 16, ss = slice_steps(k_tiles), n_sl = n_slices(k_tiles);
  const int slice_k = kStepTiles * ss * 16, xs_stride = staged_row_words(k_tiles, kDup);
  // grid: x = group of column blocks, y = row block * n_sl + k-slice, z = member (one row
  // block, the decode case, needs no division)
  const int cb = kGroup ? blockIdx.x * group : blockIdx.x;
  const int sl = (int)gridDim.y == n_sl ? (int)blockIdx.y : (int)blockIdx.y % n_sl;
  const int64_t r0 = (int64_t)((int)gridDim.y == n_sl ? 0 : (int)blockIdx.y / n_sl) * pass_rows;
  const int nr = (int)min<int64_t>(pass_rows, rows - r0);
  const int member = blockIdx.z;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;

  // (a group's first ring words are in flight while the rows are staged)
  SliceStream<K, PD> S;
  if constexpr (kGroup)
    S.start((const uint32_t *)trellis.p[member], k_tiles, tiles_n, sl * kStepTiles * ss, cb * 4 + wave);
  if (rotate) {
    // x, not xhat: the input Hadamard of the slice's 128-blocks (member's suh), in the
    // workgroup, kBatch blocks per wave at a time with every load issued first
    constexpr int kBatch = 4;
    const uint16_t *xr = xhat + member * x_member_stride + r0 * in + sl * slice_k + 2 * lane;
    const uint16_t *su = (const uint16_t *)suh.p[member] + sl * slice_k + 2 * lane;
    // blocks per row: slice_k / 128 = ss / 2, a power of two
    const int nblk = slice_k / 128, nblk_lg = __builtin_ctz(nblk), items = nr * nblk;
    for (int b0 = wave; b0 < items; b0 += 4 * kBatch) {
      uint32_t hx[kBatch], sx[kBatch];
#pragma unroll
      for (int q = 0; q < kBatch; ++q) {
        const int bi = min(b0 + 4 * q, items - 1);
        hx[q] = *reinterpret_cast<const uint32_t *>(xr + (int64_t)(bi >> nblk_lg) * in +
                                                    (bi & (nblk - 1)) * 128);
        sx[q] = *reinterpret_cast<const uint32_t *>(su + (bi & (nblk - 1)) * 128);
      }
#pragma unroll
      for (int q = 0; q < kBatch; ++q) {
        const int bi = b0 + 4 * q;
        if (bi < items) {
          float v0 = f16_to_f32((uint16_t)(hx[q] & 0xffffu)), v1 = f16_to_f32((uint16_t)(hx[q] >> 16));
          wave_had_pre(v0, v1, f16_to_f32((uint16_t)(sx[q] & 0xffffu)), f16_to_f32((uint16_t)(sx[q] >> 16)));
          stage_pair<kDup>(xs + (bi >> nblk_lg) * xs_stride, bi & (nblk - 1), lane,
                           pack_f16x2(v0, v1));
        }
      }
    }
  } else {
    // xhat rows: pair w of a k-tile (k-rows 2w, 2w + 1) to its staged position
    const uint16_t *xm = xhat + member * x_member_stride + r0 * in + sl * slice_k;
    const int pr_row = slice_k / 2, pr_lg = __builtin_ctz(pr_row);  // pairs per row
    for (int i = threadIdx.x; i < nr * pr_row; i += 256) {
      const int r = i >> pr_lg, w = i & (pr_row - 1);
      const uint32_t v = reinterpret_cast<const uint32_t *>(xm + (int64_t)r * in)[w];
      const int pw = (w & ~7) + xpos(w & 7);  // plain staged word
      if constexpr (kDup) {
        *reinterpret_cast<u32x2 *>(xs + r * xs_stride + 2 * pw) = u32x2{dup_lo(v), dup_hi(v)};
      } else {
        xs[r * xs_stride + pw] = v;
      }
    }
  }
  __syncthreads();
  // (one block: the output pointer is formed after the decode loop; formed before it, it changed
  // the loop's schedule, 2048 x 12288 K3 at 17 rows 16.2 to 16.6 us)
  if constexpr (kGroup) {
    float *p = part + (((int64_t)member * n_sl + sl) * rows + r0) * out + cb * 128 + wave * 32;
    qmv_slice_items<K, CB, PD>(S, ss, min(group, out / 128 - cb), xs + min(lane & 15, nr - 1) * xs_stride,
                               slots + wave * slot_chunks(K), [=](int it, const f32x4 &D0, const f32x4 &D1) {
                                 qmv_store(p + it * 128, out, nr, D0, D1);
                               });
  } else {
    f32x4 D0, D1;
    qmv_slice<K, CB, PD>((const uint32_t *)trellis.p[member], k_tiles, tiles_n, sl * kStepTiles * ss, cb * 4 + wave,
                         ss, xs + min(lane & 15, nr - 1) * xs_stride, slots + wave * slot_chunks(K), D0, D1);
    float *p = part + (((int64_t)member * n_sl + sl) * rows + r0) * out + cb * 128 + wave * 32;
    qmv_store(p, out, nr, D0, D1);
  }
}

// The rows of calls that take k_qmv_rows: member m's input Hadamard of every row (suh) or,
// rotate = 0, the rows as they are, in the staged k order (stage_pair). One wave per (member,
// row, kStageBatch blocks of 128), their butterfly stages interleaved.
constexpr int kStageBatch = 8;

// Bound by memory: 1000 rows of 8192 are 33 MB in and out.
__global__ __launch_bounds__(256) void k_stage_rows(const uint16_t *__restrict__ x, int64_t x_member_stride,
                                                    int64_t rows, int in, int n, exl3h::PtrTable suh, int rotate,
                                                    uint16_t *__restrict__ xrot) {
  const int lane = threadIdx.x & 63, nblk = in / 128, per_row = (nblk + kStageBatch - 1) / kStageBatch;
  const int64_t gw = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (gw >= (int64_t)n * rows * per_row) return;
  const int b0 = (int)(gw % per_row) * kStageBatch;
  const int64_t mr = gw / per_row, row = mr % rows;
  const int member = (int)(mr / rows);
  const uint16_t *xr = x + member * x_member_stride + row * in + 2 * lane;
  const uint16_t *su = (const uint16_t *)suh.p[member] + 2 * lane;
  uint32_t *out = reinterpret_cast<uint32_t *>(xrot + mr * in);
  uint32_t hx[kStageBatch];
#pragma unroll
  for (int q = 0; q < kStageBatch; ++q) hx[q] = *reinterpret_cast<const uint32_t *>(xr + min(b0 + q, nblk - 1) * 128);
  if (rotate) {
    float v0[kStageBatch], v1[kStageBatch], s0[kStageBatch], s1[kStageBatch];
#pragma unroll
    for (int q = 0; q < kStageBatch; ++q) {
      const uint32_t sx = *reinterpret_cast<const uint32_t *>(su + min(b0 + q, nblk - 1) * 128);
      v0[q] = f16_to_f32((uint16_t)(hx[q] & 0xffffu));
      v1[q] = f16_to_f32((uint16_t)(hx[q] >> 16));
      s0[q] = f16_to_f32((uint16_t)(sx & 0xffffu));
      s1[q] = f16_to_f32((uint16_t)(sx >> 16));
    }
    wave_had_pre_n<kStageBatch>(v0, v1, s0, s1);
#pragma unroll
    for (int q = 0; q < kStageBatch; ++q) hx[q] = pack_f16x2(v0[q], v1[q]);
  }
#pragma unroll
  for (int q = 0; q < kStageBatch; ++q)
    if (b0 + q < nblk) stage_pair<false>(out, b0 + q, lane, hx[q]);
}

// One wave per (member, row, 128-column block): slice partials summed in slice order,
// then the raw f32 result or the output Hadamard.
__global__ __launch_bounds__(256) void k_qmv_finalize(int n, int n_sl, int64_t rows, int out,
                                                      const float *__restrict__ part,
                                                      float *__restrict__ y32,
                                                      uint16_t *__restrict__ y16,
                                                      exl3h::PtrTable svh) {
  const int lane = threadIdx.x & 63;
  const int64_t gw = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n_cb = out / 128;
  if (gw >= (int64_t)n * rows * n_cb) return;
  const int cb = (int)(gw % n_cb);
  const int64_t rest = gw / n_cb;
  const int64_t row = rest % rows;
  const int member = (int)(rest / rows);
  const int c = cb * 128 + 2 * lane;
  const float *p = part + ((int64_t)member * n_sl * rows + row) * out + c;
  // slice partials summed in slice order; the loads of 8 slices are issued together
  float v0 = 0.0f, v1 = 0.0f;
  for (int s0 = 0; s0 < n_sl; s0 += 8) {
    float2 v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
      v[s] = *reinterpret_cast<const float2 *>(p + (int64_t)min(s0 + s, n_sl - 1) * rows * out);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s0 + s == 0) {
        v0 = v[0].x;
        v1 = v[0].y;
      } else if (s0 + s < n_sl) {
        v0 += v[s].x;
        v1 += v[s].y;
      }
    }
  }
  const int64_t o = ((int64_t)member * rows + row) * out + c;
  if (y32) {
    y32[o] = v0;
    y32[o + 1] = v1;
    return;
  }
  const uint16_t *sv = (const uint16_t *)svh.p[member] + c;
  wave_had_post(v0, v1, f16_to_f32(sv[0]), f16_to_f32(sv[1]));
  y16[o] = f32_to_f16(v0);
  y16[o + 1] = f32_to_f16(v1);
}

}  // namespace

namespace exl3h {

exl3_status launch_decode(const exl3_trellis_desc &w, uint16_t *w_hat, hipStream_t st) {
  const int tiles_n = w.out_features / 16, tiles_k = w.in_features / 16;
  dim3 grid(tiles_n, tiles_k);
  const uint32_t *t = (const uint32_t *)w.trellis;
  switch (w.codebook) {
    case 0: k_decode<0><<<grid, 256, 0, st>>>(t, w.K, tiles_n, w.out_features, w_hat); break;
    case 1: k_decode<1><<<grid, 256, 0, st>>>(t, w.K, tiles_n, w.out_features, w_hat); break;
    default: k_decode<2><<<grid, 256, 0, st>>>(t, w.K, tiles_n, w.out_features, w_hat); break;
  }
  EXL3_LAUNCHED("k_decode");
  return EXL3_OK;
}

template <int K>
static void reconstruct_cb(const exl3_trellis_desc &w, uint16_t *w_out, hipStream_t st) {
  const dim3 grid(w.out_features / 128, w.in_features / 128);
  const uint32_t *t = (const uint32_t *)w.trellis;
  const int tiles_n = w.out_features / 16, out = w.out_features;
  switch (w.codebook) {
    case 0: k_reconstruct<K, 0><<<grid, 256, 0, st>>>(t, tiles_n, out, w.suh, w.svh, w_out); break;
    case 1: k_reconstruct<K, 1><<<grid, 256, 0, st>>>(t, tiles_n, out, w.suh, w.svh, w_out); break;
    default: k_reconstruct<K, 2><<<grid, 256, 0, st>>>(t, tiles_n, out, w.suh, w.svh, w_out);
  }
}

exl3_status launch_reconstruct(const exl3_trellis_desc &w, uint16_t *w_out, hipStream_t st) {
  switch (w.K) {
    case 1: reconstruct_cb<1>(w, w_out, st); break;
    case 2: reconstruct_cb<2>(w, w_out, st); break;
    case 3: reconstruct_cb<3>(w, w_out, st); break;
    case 4: reconstruct_cb<4>(w, w_out, st); break;
    case 5: reconstruct_cb<5>(w, w_out, st); break;
    case 6: reconstruct_cb<6>(w, w_out, st); break;
    case 7: reconstruct_cb<7>(w, w_out, st); break;
    default: reconstruct_cb<8>(w, w_out, st);
  }
  EXL3_LAUNCHED("k_reconstruct");
  return EXL3_OK;
}

exl3_status launch_hadamard(const uint16_t *x16, const float *x32, int64_t rows, int n,
                            const PtrTable &s, int64_t rows_per_member, uint16_t *y,
                            hipStream_t st) {
  const int64_t waves = rows * (n / 128);
  if (waves == 0) return EXL3_OK;
  k_hadamard<<<(unsigned)((waves + 3) / 4), 256, 0, st>>>(x16, x32, rows, n, s, rows_per_member, y);
  EXL3_LAUNCHED("k_hadamard");
  return EXL3_OK;
}

template <int K, int CB, int PD>
static void qmv_go(dim3 grid, hipStream_t st, const PtrTable &tr, int tiles_n, int in, int out,
                   const uint16_t *xhat, int64_t xs, int64_t rows, int pass_rows, int group,
                   float *part, const PtrTable *suh) {
  // the wave slots and pass_rows staged rows (at most 16 x 2 KB + 8 KB: under the 64 KB
  // that a launch gets without an attribute)
  static_assert((size_t)4 * slot_chunks(8) * 16 +
                    (size_t)kPassRows * (kMaxSliceSteps * kStepTiles * tile_words(true) + 4) * 4 <=
                64 * 1024,
                "k_qmv LDS");
  const size_t lds = (size_t)4 * slot_chunks(K) * 16 +
                     (size_t)pass_rows * staged_row_words(in / 16, dup_cb(CB)) * 4;
  const auto k = group > 1 ? k_qmv<K, CB, PD, true> : k_qmv<K, CB, PD, false>;
  k<<<grid, 256, lds, st>>>(tr, tiles_n, in, out, xhat, xs, rows, pass_rows, part, suh ? *suh : PtrTable{},
                            suh ? 1 : 0, group);
}

template <int K, int CB>
static void qmv_pd(int pd, dim3 grid, hipStream_t st, const PtrTable &tr, int tiles_n, int in,
                   int out, const uint16_t *xhat, int64_t xs, int64_t rows, int pass_rows, int group,
                   float *part, const PtrTable *suh) {
  if (pd == 1)
    return qmv_go<K, CB, 1>(grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh);
  if constexpr (K <= 4) {
    if (pd >= 4)
      return qmv_go<K, CB, 4>(grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh);
  }
  qmv_go<K, CB, 2>(grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh);
}

template <int K>
static void qmv_cb(int cb, int pd, dim3 grid, hipStream_t st, const PtrTable &tr, int tiles_n,
                   int in, int out, const uint16_t *xhat, int64_t xs, int64_t rows, int pass_rows, int group,
                   float *part, const PtrTable *suh) {
  switch (cb) {
    case 0: qmv_pd<K, 0>(pd, grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh); break;
    case 1: qmv_pd<K, 1>(pd, grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh); break;
    case 2: qmv_pd<K, 2>(pd, grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh); break;
    case 3: qmv_pd<K, 3>(pd, grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh); break;
    default: qmv_pd<K, 4>(pd, grid, st, tr, tiles_n, in, out, xhat, xs, rows, pass_rows, group, part, suh); break;
  }
}

int qmv_pass_rows(int64_t rows) {
  const exl3_tuning tn = tuning();
  int pr = tn.rows_per_pass > 0 ? tn.rows_per_pass : kPassRows;
  if (pr > kPassRows) pr = kPassRows;
  return (int)std::min<int64_t>(pr, std::max<int64_t>(rows, 1));
}

int qmv_slices(int in) { return n_slices(in / 16); }

// Waves of k_stage_rows.
static int64_t stage_waves(int64_t rows, int in, int n) {
  return (int64_t)n * rows * ((in / 128 + kStageBatch - 1) / kStageBatch);
}

// The linear's path: the slice-parallel k_qmv (16 rows per decode, f32 slice partials through
// memory, the rotation repeated by every column block) or k_qmv_rows (64 or 128 rows per
// decode, the whole k range in one workgroup) in one of its three shapes, whichever is
// estimated faster. The estimates, in us, follow measurements at K = 4 (mcg) over in 640 to
// 12288, out 1024 to 24576 and 17 to 1024 rows: the slice path takes 4.0 per 16 rows and
// 2^24 weights; a workgroup of k_qmv_rows takes 27 (64 x 128 outputs), 42 (128 x 128) or 79
// (128 x 256) per 4096 of k while every CU has one, and 35, 46 or 65 when it is alone.
// 4096 x 4096, slice path against the estimate's choice: 38 against 38 at 128 rows, 68
// against 43 at 256, 258 against 60 at 1024; 4096 x 24576: 44 against 40 at 17 rows, 1586
// against 241 at 1024; 8192 x 4096 at 1000 rows: 495 against 101. Calls of up to 16 rows (one
// decode either way) keep the slice path. rb = 0: the slice path.
RowsPlan rows_plan(int in, int out, int64_t rows, int n) {
  RowsPlan best{};
  // (calls past the slice path's grid limit are refused there)
  if (rows <= 16 || (int64_t)n_slices(in / 16) * ((rows + 15) / 16) > 65535) return best;
  // k_stage_rows' grid: a launch has at most 2^32 - 1 threads in a dimension (128 members of
  // 1536 x 128 pass it from 262,144 rows, where the slice path's launches still fit)
  if (stage_waves(rows, in, n) * 64 > (int64_t)UINT32_MAX - 256) return best;
  const double k = in / 4096.0;
  double t_best = 4.0 + 4.0 * (double)((rows + 15) / 16) * ((double)in * out * n / (1 << 24));
  const struct {
    int rb, waves;
    double alone, full;
  } shapes[] = {{4, 4, 35, 27}, {8, 4, 46, 42}, {8, 8, 65, 79}};
  for (const auto &s : shapes) {
    const int64_t tiles = (rows + 16 * s.rb - 1) / (16 * s.rb);
    const int64_t wgs = tiles * ((out / 32 + s.waves - 1) / s.waves) * n;
    if (wgs * s.waves * 64 > (int64_t)UINT32_MAX) continue;
    const double t = 8.0 + k * std::max(s.alone, s.full * (double)((wgs + 255) / 256));
    if (t < t_best) {
      t_best = t;
      best = RowsPlan{s.rb, s.waves};
    }
  }
  return best;
}

exl3_status launch_stage_rows(const uint16_t *x, int64_t x_member_stride, int64_t rows, int in, int n,
                              const PtrTable *suh, uint16_t *xrot, hipStream_t st) {
  const int64_t waves = stage_waves(rows, in, n);
  k_stage_rows<<<(unsigned)((waves + 3) / 4), 256, 0, st>>>(x, x_member_stride, rows, in, n, suh ? *suh : PtrTable{},
                                                            suh ? 1 : 0, xrot);
  EXL3_LAUNCHED("k_stage_rows");
  return EXL3_OK;
}

exl3_status launch_qmv_rows(const exl3_trellis_desc &shape, const RowsPlan &p, const PtrTable &trellis, int n,
                            const uint16_t *xrot, int64_t rows, float *y32, uint16_t *y16, const PtrTable &svh,
                            hipStream_t st) {
  exl3d::RowsArgs a{};
  a.xrot = xrot;
  a.rows = rows;
  a.in = shape.in_features;
  a.out = shape.out_features;
  a.row_tiles = (int)((rows + 16 * p.rb - 1) / (16 * p.rb));
  a.col_groups = (a.out / 32 + p.waves - 1) / p.waves;
  a.members = n;
  a.y32 = y32;
  a.y16 = y16;
  a.trellis = trellis;
  a.svh = svh;
  if (shape.K <= 4) launch_qmv_rows_k14(shape.K, shape.codebook, p.rb, p.waves, a, st);
  else launch_qmv_rows_k58(shape.K, shape.codebook, p.rb, p.waves, a, st);
  EXL3_LAUNCHED("k_qmv_rows");
  return EXL3_OK;
}

// Column blocks per workgroup of k_qmv (1, 2 or 4) from the call's one-block workgroups and rows
// a pass: the fewest rounds of 256 CUs times a workgroup's work, g blocks' decode and one
// rotation (rows / 32 of a block's decode). The rounds weigh most: 4096 x 50176 (K4, 3136
// workgroups) at 1 row takes 32.4, 34.0, 38.3 us with 1, 2, 4 blocks (13, 7, 4 rounds). At least
// 768 workgroups stay (3 per CU), and below 8 rows, whose rotation is cheap, 2048 (more than are
// resident at once): 4096 x 32768 (K4, 2048) 22.5, 23.4, 24.9 at 1 row, 30.7, 30.2, 28.3 at 8;
// 4096 x 24576 (K4, 1536) 33.3, 30.3, 29.6 at 16; 8192 x 24576 (K3, 3072) 41.5, 39.8, 35.1 at 8;
// the 4096 x 154880 head (K6, 9680) 96, 94, 94 at 1 row, 110, 104, 104 at 4, 133, 122, 119 at 8.
static int qmv_group(int64_t blocks, int rows) {
  int best = 1;
  double t_best = 0;
  for (int g = 1; g <= 4; g *= 2) {
    const int64_t wgs = (blocks + g - 1) / g;
    if (g > 1 && wgs < (rows < 8 ? 2048 : 768)) break;
    const double t = (double)((wgs + 255) / 256) * (g + rows / 32.0);
    if (g == 1 || t < t_best) {
      t_best = t;
      best = g;
    }
  }
  return best;
}

exl3_status launch_qmv(const exl3_trellis_desc &shape, const PtrTable &trellis, int n,
                       const uint16_t *xhat, int64_t x_member_stride, int64_t rows, float *part,
                       hipStream_t st, const PtrTable *suh) {
  const int in = shape.in_features, out = shape.out_features;
  const int k_tiles = in / 16;
  const int pr = qmv_pass_rows(rows);
  const int64_t gy = (int64_t)n_slices(k_tiles) * ((rows + pr - 1) / pr);
  if (gy > 65535 || n > 65535) return fail(EXL3_ERR_UNSUPPORTED, "linear launch too large");
  const int group = qmv_group((int64_t)(out / 128) * gy * n, pr);
  dim3 grid((unsigned)((out / 128 + group - 1) / group), (unsigned)gy, (unsigned)n);
  const int tiles_n = out / 16, pd = prefetch_steps(k_tiles, shape.K);
  // the weight form of the process-wide tuning (the reference's f16 weights by default)
  const int kcb = kernel_cb(shape.codebook, tuning().weight_form);
  switch (shape.K) {
#define EXL3_K(KK)                                                                        \
  case KK:                                                                                \
    qmv_cb<KK>(kcb, pd, grid, st, trellis, tiles_n, in, out, xhat, x_member_stride, rows, \
               pr, group, part, suh);                                                     \
    break;
    EXL3_K(1) EXL3_K(2) EXL3_K(3) EXL3_K(4) EXL3_K(5) EXL3_K(6) EXL3_K(7) EXL3_K(8)
#undef EXL3_K
    default: return fail(EXL3_ERR_INVALID, "K out of range");
  }
  EXL3_LAUNCHED("k_qmv");
  return EXL3_OK;
}

exl3_status launch_qmv_finalize(int n, int n_sl, int64_t rows, int out, const float *part,
                                float *y32, uint16_t *y16, const PtrTable &svh, hipStream_t st) {
  const int64_t waves = (int64_t)n * rows * (out / 128);
  if (waves == 0) return EXL3_OK;
  k_qmv_finalize<<<(unsigned)((waves + 3) / 4), 256, 0, st>>>(n, n_sl, rows, out, part, y32,
                                                              y16, svh);
  EXL3_LAUNCHED("k_qmv_finalize");
  return EXL3_OK;
}

}  // namespace exl3h
