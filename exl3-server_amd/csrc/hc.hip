// The steps either side of the MoE in the GLM-5 batch step (glm5_forward.cpp:434-438):
// the hyper-connection prepare (g5_hc_prepare, glm5_hc.cpp:242-340), the RMSNorm of its
// collapsed stream (rms_norm, glm5_attn.cpp:12-22) and the hyper-connection mix
// (g5_hc_mix, glm5_hc.cpp:342-355), gfx950.
//
//  k_hc_proj      grid (slice of the N*D axis, tile of positions): the slice's part of the
//                 W = (2+N)*N projections x . fn[j] (fn stored (W, N*D), as the reference's
//                 F.linear weight) on the f32 matrix instruction, and of the sum of
//                 squares; f32 partials per slice.
//  k_hc_finalize  two kinds of workgroups side by side, which sum the partials in order and
//                 take the RMS factor (w = rms * x.fn, the fused reference kernel's
//                 per-term product folded out of the sum): one per position forms pre and
//                 the collapsed stream sum_n pre[n] * streams[n] rounded to f16 (and,
//                 given a norm weight, the RMSNorm of that row fused behind it); one per
//                 few positions forms post and comb, with the softmax over the last axis
//                 and the Sinkhorn in the reference's loop order (glm5_hc.cpp:321-324).
//  k_rms_norm     the RMSNorm alone, one workgroup per row.
//  k_hc_mix       post[n] * out + comb^T @ residual in f16 (also fused into the MoE
//                 combine, which then writes the new streams directly).
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>
#include <type_traits>

#include "exl3_device.hpp"
#include "exl3_internal.hpp"
#include "exl3_moe.h"
#include "moe_common.hpp"

using namespace exl3d;

namespace {

constexpr int kHcMaxN = 8;                       // streams (W <= 80)
constexpr int kHcMaxD = 8192;
static_assert(kHcMaxN <= exl3m::kHcMixMax, "the mix's residual registers");
constexpr int kHcNarrowN = 4;                    // the narrow kernels' streams (W <= 24; GLM-5's 4)
// The projections' sums over the N*D axis: chunks of 64 elements (each from zero), groups of
// 4 chunks, super-groups of 4 groups, each level's sums added in order. Calls of few
// positions write the groups' sums, of many the super-groups'; the finalize adds up the
// rest, so a position's results do not depend on how many the call has.
constexpr int kHcChunk = 64;
constexpr int kHcWaves = 4;       // per projection workgroup: a group's chunks or a super-group's groups
constexpr int kHcFan = 4;         // chunks per group, groups per super-group
static_assert(kHcWaves == kHcFan, "a wave per chunk or per group");
constexpr int kHcRows = 16;       // positions per row tile (the MFMA's rows)
// Positions from which a projection wave takes a group of chunks instead of one (4 streams of
// 4096, both kernels of the prepare, kernel trace): 15.3 us with a chunk against 16.8 with a
// group at 256 positions, 17.9 against 17.7 at 384, 68 against 47 at 2048; at 64, 10.6 against
// 15.1. (256 positions of one 512-wide stream: 9.0 against 10.9.)
constexpr int kHcManyRows = 384;
// Calls of few positions and more than 4 streams: a wave's chunk is 48 to 80 dependent-issue
// MFMAs (3 to 5 tiles of projections). While the call has at most this many workgroups of all
// tiles, one per CU, each tile gets a workgroup of its own. Both kernels, 8 streams: 11.5 us
// against 9.5 at one position of 1024 (32 workgroups), 22.6 against 21.6 at 16 of 8192 (256),
// but 19.8 against 20.7 at 64 of 4096 (512); 5 streams of 512 at 383 positions (240) 11.1 either
// way. (A thread per projection, before: 10.4 at one position of 8 x 1024.)
constexpr int kHcSplitGroups = 256;

// Values per (position, partial): the W = (2+N)*N projections' bound (kN = 4: 1..4
// streams; kN = 8: 5..8), then the sum of squares at index kMaxW.
template <int kN>
struct HcShape {
  static constexpr int kMaxW = (2 + kN) * kN;
  static constexpr int kVals = kMaxW + 1;
  static constexpr int kPos = kN <= kHcNarrowN ? 8 : 3;  // positions per post/comb workgroup
  static_assert(kPos * kVals <= 256, "a thread per value");
};
// Values per partial for N streams (the part buffer's layout).
constexpr int hc_vals(int N) { return N <= kHcNarrowN ? HcShape<kHcNarrowN>::kVals : HcShape<kHcMaxN>::kVals; }
constexpr int hc_slices(int ND, int chunks) { return (ND / kHcChunk + chunks - 1) / chunks; }

__device__ __forceinline__ float wave_sum(float v) {
  v += xor_lanes<1>(v);
  v += xor_lanes<2>(v);
  v += xor_lanes<4>(v);
  v += xor_lanes<8>(v);
  v += xor_lanes<16>(v);
  v += xor_lanes<32>(v);
  return v;
}

__device__ __forceinline__ float h2f(uint16_t v) { return (float)bitcast<f16>(v); }

// The projections x . fn[j] of 16 positions on the f32 matrix instruction
// (v_mfma_f32_16x16x4_f32: 16 positions x 16 projections x 4 k), NT tiles of 16 projections.
// Lane l: position (A) or projection (B) l % 16, k group l / 16; of every 32 k it holds the 8
// consecutive ones of its group, so a chunk is two 16-byte loads of the position's streams
// and four of each fn row, and MFMA j of a 32-k step takes element j of every group. The
// sum of squares is one fma per element beside them.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));  // streams: 8-byte aligned
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int NT, int RT>
struct HcChunkRegs {
  u32x4 a[RT][2];
  f32x4 b[NT][2][2];
};

// srow / frow[t]: this lane's positions and projections at its k group.
template <int NT, int RT>
__device__ __forceinline__ void hc_load(const uint16_t *const (&srow)[RT], const float *const (&frow)[NT], int k0,
                                        HcChunkRegs<NT, RT> &c) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int r = 0; r < RT; ++r) c.a[r][q] = *reinterpret_cast<const u32x4_a8 *>(srow[r] + k0 + 32 * q);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      c.b[t][q][0] = *reinterpret_cast<const f32x4 *>(frow[t] + k0 + 32 * q);
      c.b[t][q][1] = *reinterpret_cast<const f32x4 *>(frow[t] + k0 + 32 * q + 4);
    }
  }
}

// One chunk from zero of RT row tiles.
template <int NT, int RT>
__device__ __forceinline__ void hc_chunk(const HcChunkRegs<NT, RT> &c, f32x4 (&E)[RT][NT], float (&sq)[RT]) {
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    sq[r] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) E[r][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const float x = h2f((uint16_t)(c.a[r][q][j >> 1] >> (16 * (j & 1))));
        sq[r] = fmaf(x, x, sq[r]);
#pragma unroll
        for (int t = 0; t < NT; ++t)
          E[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, c.b[t][q][j >> 2][j & 3], E[r][t], 0, 0, 0);
      }
}

// Bound by the matrix unit and the stream reads together: 2048 positions of 4 x 4096 are 1.05 M
// 16x16x4 products (3/4 of their columns used; 13.7 us at 32 cycles each) over 67 MB (13 us at
// the 5.1 TB/s of a copy). Measured there: 30.8 us, where a thread per projection, reading its
// own row of the streams, took 474; two row tiles per wave, so that a loaded fn value serves 32
// positions: 30.8 against 36 for one, and 33 for four (one wave per SIMD). At 4 positions both
// forms are a round of loads: 4.6 us.
// Workgroup (slice, RT row tiles, tiles of projections from NT * blockIdx.z): 4 waves of kC
// consecutive chunks each (kC = 1: the slice is a group; kC = 4: a super-group), every chunk's
// loads issued one chunk ahead, then the waves' sums added in order through LDS.
template <int kN, int NT, int RT, int kC>
__global__ __launch_bounds__(64 * kHcWaves) void k_hc_proj(const uint16_t *__restrict__ streams, int64_t P, int ND,
                                                           int W, const float *__restrict__ fn,
                                                           float *__restrict__ part) {
  static_assert(kC == 1 || kC == kHcFan, "a wave's chunks: one, or a group");
  __shared__ f32x4 s_d[kHcWaves][RT][NT][64];
  __shared__ float s_q[kHcWaves][RT][64];
  constexpr int kVals = HcShape<kN>::kVals;
  const int slice = blockIdx.x, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p0 = (int64_t)blockIdx.y * (kHcRows * RT);
  const int j0 = 16 * NT * (int)blockIdx.z;  // this workgroup's first projection
  const int chunks = ND / kHcChunk;
  const int c0 = (slice * kHcWaves + wave) * kC;
  const int n = min(kC, chunks - c0);                                          // this wave's chunks
  const int n_waves = min(kHcWaves, (chunks - slice * kHcWaves * kC + kC - 1) / kC);  // waves with chunks
  // this lane's positions and projections at its k group (rows past P read the last one,
  // projections past W the last one: neither is stored)
  const uint16_t *srow[RT];
  const float *frow[NT];
#pragma unroll
  for (int r = 0; r < RT; ++r) srow[r] = streams + min<int64_t>(p0 + 16 * r + c, P - 1) * ND + 8 * g;
#pragma unroll
  for (int t = 0; t < NT; ++t) frow[t] = fn + (int64_t)min(j0 + 16 * t + c, W - 1) * ND + 8 * g;
  f32x4 D[RT][NT];
  float sq[RT];
  if (n > 0) {
    HcChunkRegs<NT, RT> r[2];
    hc_load<NT, RT>(srow, frow, c0 * kHcChunk, r[0]);
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      if (i + 1 < kC) hc_load<NT, RT>(srow, frow, (c0 + min(i + 1, n - 1)) * kHcChunk, r[(i + 1) & 1]);
      f32x4 E[RT][NT];
      float eq[RT];
      hc_chunk<NT, RT>(r[i & 1], E, eq);
#pragma unroll
      for (int rr = 0; rr < RT; ++rr) {
        if (i == 0) {
          sq[rr] = eq[rr];
#pragma unroll
          for (int t = 0; t < NT; ++t) D[rr][t] = E[rr][t];
        } else if (i < n) {
          sq[rr] = sq[rr] + eq[rr];
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int k = 0; k < 4; ++k) D[rr][t][k] = D[rr][t][k] + E[rr][t][k];
        }
      }
    }
#pragma unroll
    for (int rr = 0; rr < RT; ++rr) {
#pragma unroll
      for (int t = 0; t < NT; ++t) s_d[wave][rr][t][lane] = D[rr][t];
      // a group's squares: each k group's over the chunks (here, or over the waves below),
      // then the four k groups'
      if constexpr (kC > 1) {
        sq[rr] = sq[rr] + xor_lanes<16>(sq[rr]);
        sq[rr] = sq[rr] + xor_lanes<32>(sq[rr]);
      }
      s_q[wave][rr][lane] = sq[rr];
    }
  }
  __syncthreads();
  // the (row tile, projection tile) sums over the waves, one pair per wave at a time; lane l
  // holds projection 16t + l % 16 of positions 4 (l / 16) + i
  for (int o = wave; o < RT * NT; o += kHcWaves) {
    const int rr = o / NT, t = o % NT;
    f32x4 v = s_d[0][rr][t][lane];
    for (int w = 1; w < n_waves; ++w) {
      const f32x4 u = s_d[w][rr][t][lane];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = v[k] + u[k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t p = p0 + 16 * rr + 4 * g + k;
      if (p < P && j0 + 16 * t + c < W) part[(p * gridDim.x + slice) * kVals + j0 + 16 * t + c] = v[k];
    }
  }
  if (wave < RT && j0 == 0) {
    float v = s_q[0][wave][lane];
    for (int w = 1; w < n_waves; ++w) v = v + s_q[w][wave][lane];
    if constexpr (kC == 1) {
      v = v + xor_lanes<16>(v);
      v = v + xor_lanes<32>(v);
    }
    const int64_t p = p0 + 16 * wave + c;
    if (g == 0 && p < P) part[(p * gridDim.x + slice) * kVals + HcShape<kN>::kMaxW] = v;
  }
}

// A value of one position from its partials pp[slice * kVals], the super-groups' sums (calls
// of many positions), in order.
template <int kVals>
__device__ __forceinline__ float hc_value(const float *pp, int n_slices) {
  constexpr int kB = 16;  // loads in flight
  float acc = 0.0f;
  for (int c0 = 0; c0 < n_slices; c0 += kB) {
    float v[kB];
#pragma unroll
    for (int q = 0; q < kB; ++q) v[q] = pp[min(c0 + q, n_slices - 1) * kVals];
#pragma unroll
    for (int q = 0; q < kB; ++q)
      if (c0 + q < n_slices) acc = c0 + q == 0 ? v[0] : acc + v[q];
  }
  return acc;
}

// Calls of few positions: one position's values j(i), i < nv, from the groups' partials
// pp[group * kVals]. Thread (super-group, value) adds its super-group's 4 partials in order
// (one round of loads for the whole workgroup: hc_super_load, then other loads may follow,
// then hc_super_sum), and the super-groups' sums are added in order from LDS.
constexpr int kHcMaxSupers = kHcMaxN * kHcMaxD / (kHcChunk * kHcFan * kHcFan);
template <int kVals, typename J>
__device__ __forceinline__ void hc_super_load(const float *pp, int n_groups, int nv, J &&j, int item, float (&v)[kHcFan]) {
  const int s = item / nv, at = j(item % nv);
#pragma unroll
  for (int q = 0; q < kHcFan; ++q) v[q] = pp[min(s * kHcFan + q, n_groups - 1) * kVals + at];
}
template <int kVals, typename J>
__device__ __forceinline__ void hc_super_sum(const float *pp, int n_groups, int nv, J &&j, float (&v)[kHcFan],
                                             float *sup, float *vals) {
  const int ns = (n_groups + kHcFan - 1) / kHcFan, items = ns * nv;
  for (int item = threadIdx.x; item < items; item += 256) {
    if (item >= 256) hc_super_load<kVals>(pp, n_groups, nv, j, item, v);
    const int n = n_groups - item / nv * kHcFan;
    float t = v[0];
#pragma unroll
    for (int q = 1; q < kHcFan; ++q)
      if (q < n) t += v[q];
    sup[item] = t;
  }
  __syncthreads();
  if ((int)threadIdx.x < nv) {
    float acc = sup[threadIdx.x];
    for (int s = 1; s < ns; ++s) acc += sup[s * nv + threadIdx.x];
    vals[j(threadIdx.x)] = acc;
  }
  __syncthreads();
}

// Sum of one value over a workgroup of 4 waves, the waves' sums added in wave order.
__device__ __forceinline__ float block_sum(float v, float *red) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  const float t = ((red[0] + red[1]) + red[2]) + red[3];
  __syncthreads();
  return t;
}

// A row of D f16 values (a multiple of 8 with streams, even for the norm alone) over a
// workgroup: thread t holds the 8 values from d = 8 * (t + 256 * i), i < kV, in 16-byte
// loads (rows are 4-byte aligned at least). The last vector of a row whose D is no
// multiple of 8 is taken pair by pair.
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ int vec_d(int i) { return 8 * ((int)threadIdx.x + 256 * i); }

__device__ __forceinline__ u32x4 load_vec(const uint16_t *row, int d, int D) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if (d + 8 <= D) {
    v = *reinterpret_cast<const u32x4_a4 *>(row + d);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (d + 2 * k < D) v[k] = *reinterpret_cast<const uint32_t *>(row + d + 2 * k);
  }
  return v;
}
__device__ __forceinline__ void store_vec(uint16_t *row, int d, int D, const u32x4 &v) {
  if (d + 8 <= D) {
    *reinterpret_cast<u32x4_a4 *>(row + d) = v;
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (d + 2 * k < D) *reinterpret_cast<uint32_t *>(row + d + 2 * k) = v[k];
  }
}
__device__ __forceinline__ float vec_el(const u32x4 &v, int e) { return h2f((uint16_t)(v[e >> 1] >> (16 * (e & 1)))); }

// y = f16(f16(x * r) * w) on this thread's values (x: the row's f16 values, zeros past D;
// wv: the norm weights), r = rsqrt(mean(x^2) + eps) of the row: the thread's squares summed
// in order, then the workgroup's sum.
template <int kV>
__device__ __forceinline__ void rms_vecs(const u32x4 (&x)[kV], int D, float eps, const u32x4 (&wv)[kV], uint16_t *y,
                                         float *red) {
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kV; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = vec_el(x[i], e);
      ss = fmaf(v, v, ss);
    }
  const float total = block_sum(ss, red);
  const float r = 1.0f / sqrtf(total / (float)D + eps);
#pragma unroll
  for (int i = 0; i < kV; ++i)
    if (vec_d(i) < D) {
      u32x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float n0 = (float)to_f16(vec_el(x[i], 2 * k) * r), n1 = (float)to_f16(vec_el(x[i], 2 * k + 1) * r);
        o[k] = pack_f16x2(n0 * vec_el(wv[i], 2 * k), n1 * vec_el(wv[i], 2 * k + 1));
      }
      store_vec(y, vec_d(i), D, o);
    }
}

// post and comb of the positions p0 .. p0 + kPos - 1 (of p0 alone in a call of few positions)
// by one workgroup (the latency-bound
// Sinkhorn of a wave runs beside the other workgroups' collapse and norm).
template <int kN>
__device__ __forceinline__ void hc_comb(int64_t p0, int64_t P, int N, int W, int64_t ND, int n_slices, int fan,
                                        const float *part, const float *base, const float *scale, int iters, float eps,
                                        float *post_out, float *comb_out, float *sup) {
  using S = HcShape<kN>;
  __shared__ float vals[S::kPos][S::kVals];
  const int t = threadIdx.x;
  if (fan == 1) {
    const int r = t / S::kVals, j = t % S::kVals;
    const int64_t p = p0 + r;
    if (r < S::kPos && p < P && ((j >= N && j < W) || j == S::kMaxW))
      vals[r][j] = hc_value<S::kVals>(part + p * n_slices * S::kVals + j, n_slices);
    __syncthreads();
  } else {
    const float *pp = part + p0 * n_slices * S::kVals;
    const int nv = W - N + 1;
    auto at = [&](int i) { return i < nv - 1 ? N + i : S::kMaxW; };
    float v[kHcFan];
    hc_super_load<S::kVals>(pp, n_slices, nv, at, t, v);
    hc_super_sum<S::kVals>(pp, n_slices, nv, at, v, sup, vals[0]);
    P = p0 + 1;  // this workgroup's one position
  }
  if constexpr (kN > kHcNarrowN) {
    // a wave per position: lane l holds comb entry (l / 8, l % 8) of an 8 x 8 layout
    // (entries outside N x N stay 0): a row is 8 consecutive lanes, a column the lanes 8
    // apart; sums by lane exchanges at distances 1, 2, 4 (rows) and 8, 16, 32 (columns)
    const int r = t >> 6, lane = t & 63;
    const int64_t p = p0 + r;
    if (r >= S::kPos || p >= P) return;
    const float rms = 1.0f / sqrtf(vals[r][S::kMaxW] / (float)ND + eps);
    if (lane < N) {
      const float wq = vals[r][N + lane] * rms;
      post_out[p * N + lane] = 2.0f * (1.0f / (1.0f + expf(-(wq * scale[1] + base[N + lane]))));
    }
    const int ci = lane >> 3, cj = lane & 7;
    const bool live = ci < N && cj < N;
    auto row_sum = [&](float v) {
      const float s = v + xor_lanes<1>(v);
      const float s2 = s + xor_lanes<2>(s);
      return s2 + xor_lanes<4>(s2);
    };
    auto col_sum = [&](float v) {
      const float s = v + xor_lanes<8>(v);
      const float s2 = s + xor_lanes<16>(s);
      return s2 + xor_lanes<32>(s2);
    };
    const float z = live ? vals[r][2 * N + ci * N + cj] * rms * scale[2] + base[2 * N + ci * N + cj] : -INFINITY;
    float m = fmaxf(z, xor_lanes<1>(z));
    m = fmaxf(m, xor_lanes<2>(m));
    m = fmaxf(m, xor_lanes<4>(m));
    float c = live ? expf(z - m) : 0.0f;
    const float rs = row_sum(c);
    c = live ? c / rs + eps : 0.0f;
    auto norm = [&](float v, float sum) { return live ? v / (sum + eps) : 0.0f; };
    c = norm(c, col_sum(c));
    for (int it = 0; it < iters - 1; ++it) {
      c = norm(c, row_sum(c));
      c = norm(c, col_sum(c));
    }
    if (live) comb_out[p * N * N + ci * N + cj] = c;
  } else {
    // 16 lanes per position: lane l of them holds comb entry (l / 4, l % 4) of a 4 x 4
    // layout (entries outside N x N stay 0), so a row is a quad and a column the lanes j,
    // j + 4, j + 8, j + 12: row sums by quad-permute DPP, column sums by row-rotate DPP, no
    // LDS round trip per reduction
    const int r = t >> 4, lane = t & 15;
    const int64_t p = p0 + r;
    if (r >= S::kPos || p >= P) return;  // whole rows of 16 lanes: the DPP stays within one
    const float rms = 1.0f / sqrtf(vals[r][S::kMaxW] / (float)ND + eps);
    if (lane < N) {
      const float wq = vals[r][N + lane] * rms;
      post_out[p * N + lane] = 2.0f * (1.0f / (1.0f + expf(-(wq * scale[1] + base[N + lane]))));
    }
    const int ci = lane >> 2, cj = lane & 3;
    const bool live = ci < N && cj < N;
    auto dpp = [](float v, auto ctrl) {
      return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(ctrl)::value,
                                                                 0xF, 0xF, false));
    };
    using X1 = std::integral_constant<int, 0xB1>;   // lane ^ 1
    using X2 = std::integral_constant<int, 0x4E>;   // lane ^ 2
    using R4 = std::integral_constant<int, 0x124>;  // rotate right by 4 within 16 lanes
    using R8 = std::integral_constant<int, 0x128>;  // rotate right by 8 within 16 lanes
    auto row_sum = [&](float v) {
      const float s = v + dpp(v, X1{});
      return s + dpp(s, X2{});
    };
    auto col_sum = [&](float v) {
      const float s = v + dpp(v, R4{});
      return s + dpp(s, R8{});
    };
    // softmax over the last axis (j), then + eps
    const float z = live ? vals[r][2 * N + ci * N + cj] * rms * scale[2] + base[2 * N + ci * N + cj] : -INFINITY;
    float m = fmaxf(z, dpp(z, X1{}));
    m = fmaxf(m, dpp(m, X2{}));
    float c = live ? expf(z - m) : 0.0f;
    const float rs = row_sum(c);
    c = live ? c / rs + eps : 0.0f;
    // Sinkhorn: columns, then (iters - 1) x (rows, columns); the entries outside N x N
    // are set to 0 at every step (a padded row or column sums to 0, so at eps = 0 its
    // own division would be 0 / 0; the sums themselves run on every lane for the DPP)
    auto norm = [&](float v, float sum) { return live ? v / (sum + eps) : 0.0f; };
    c = norm(c, col_sum(c));
    for (int it = 0; it < iters - 1; ++it) {
      c = norm(c, row_sum(c));
      c = norm(c, col_sum(c));
    }
    if (live) comb_out[p * N * N + ci * N + cj] = c;
  }
}

// At 2048 positions of 4 x 4096 the streams are read once more and the rows written, 84 MB:
// 16.4 us (5.1 TB/s), from 56 with two workgroups per position, 4-byte loads and 256 partials
// a value; at 4 positions a few dependent round trips: 6.2 us, from 10.4.
// Workgroups [0, comb_blocks): post and comb of kPos positions each (calls of few
// positions, whose partials are the groups' sums, fan = kHcFan: of one); then one workgroup per
// position: pre, the collapsed stream and its norm, kV vectors of 8 values per thread.
template <int kN, int kV>
__global__ __launch_bounds__(256) void k_hc_finalize(const uint16_t *__restrict__ streams, int64_t P, int N, int D,
                                                     int W, int n_slices, int fan, int comb_blocks,
                                                     const float *__restrict__ part,
                                                     const float *__restrict__ base, const float *__restrict__ scale,
                                                     int iters, float eps, const uint16_t *__restrict__ norm_w,
                                                     float norm_eps, uint16_t *__restrict__ out,
                                                     float *__restrict__ post_out, float *__restrict__ comb_out) {
  using S = HcShape<kN>;
  constexpr bool kNarrow = kN <= kHcNarrowN;
  const int64_t ND = (int64_t)N * D;
  __shared__ float sup[kHcMaxSupers * kN / kHcMaxN * S::kVals];
  if ((int)blockIdx.x < comb_blocks) {
    hc_comb<kN>((int64_t)blockIdx.x * (fan == 1 ? S::kPos : 1), P, N, W, ND, n_slices, fan, part, base, scale, iters,
                eps, post_out, comb_out, sup);
    return;
  }
  __shared__ float pre[S::kVals];
  __shared__ float red[4];
  const int64_t p = blockIdx.x - comb_blocks;
  const int t = threadIdx.x;
  // the N pre projections' and the squares' partials (needed first, so loaded first)
  const float *pp = part + p * n_slices * S::kVals;
  auto at = [&](int i) { return i < N ? i : S::kMaxW; };
  float pv[kHcFan];
  if (fan > 1) hc_super_load<S::kVals>(pp, n_slices, N + 1, at, t, pv);
  // the row's streams, in flight while the projections are finished (the narrow variant; the
  // wide one loads each stream at the collapse, to keep its registers)
  const uint16_t *srow = streams + p * ND;
  u32x4 sp[kNarrow ? kN : 1][kV];
  if constexpr (kNarrow) {
#pragma unroll
    for (int n = 0; n < kN; ++n)
#pragma unroll
      for (int i = 0; i < kV; ++i)
        sp[n][i] = n < N ? load_vec(srow + (int64_t)n * D, vec_d(i), D) : u32x4{0u, 0u, 0u, 0u};
  }
  // the norm weights too (the row's own streams stand in when there is no norm: same
  // length, never used)
  u32x4 wv[kV];
#pragma unroll
  for (int i = 0; i < kV; ++i) wv[i] = load_vec(norm_w ? norm_w : srow, vec_d(i), D);
  if (fan > 1) {
    hc_super_sum<S::kVals>(pp, n_slices, N + 1, at, pv, sup, pre);
  } else {
    if (t <= N) pre[at(t)] = hc_value<S::kVals>(pp + at(t), n_slices);
    __syncthreads();
  }
  const float rms = 1.0f / sqrtf(pre[S::kMaxW] / (float)ND + eps);
  float pn[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n)
    pn[n] = n < N ? 1.0f / (1.0f + expf(-(pre[n] * rms * scale[0] + base[n]))) + eps : 0.0f;
  // collapsed = sum_n pre[n] * streams[n], in f16
  u32x4 x[kV];
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = 0.0f;
    if constexpr (kNarrow) {
#pragma unroll
      for (int n = 0; n < kN; ++n)
        if (n < N)
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] = fmaf(pn[n], vec_el(sp[n][i], e), a[e]);
    } else {
      u32x4 v[kN];
#pragma unroll
      for (int n = 0; n < kN; ++n) v[n] = load_vec(srow + (int64_t)min(n, N - 1) * D, vec_d(i), D);
#pragma unroll
      for (int n = 0; n < kN; ++n)
        if (n < N)
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] = fmaf(pn[n], vec_el(v[n], e), a[e]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) x[i][k] = pack_f16x2(a[2 * k], a[2 * k + 1]);
  }
  if (!norm_w) {
#pragma unroll
    for (int i = 0; i < kV; ++i)
      if (vec_d(i) < D) store_vec(out + p * D, vec_d(i), D, x[i]);
    return;
  }
  rms_vecs<kV>(x, D, norm_eps, wv, out + p * D, red);
}

template <int kV>
__global__ __launch_bounds__(256) void k_rms_norm(const uint16_t *__restrict__ xin, int D, const uint16_t *__restrict__ w,
                                                  float eps, uint16_t *__restrict__ y) {
  __shared__ float red[4];
  const int64_t p = blockIdx.x;
  u32x4 x[kV], wv[kV];
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    x[i] = load_vec(xin + p * D, vec_d(i), D);
    wv[i] = load_vec(w, vec_d(i), D);
  }
  rms_vecs<kV>(x, D, eps, wv, y + p * D, red);
}

// f(kV): the vectors of 8 values per thread of a row of D values.
template <typename F>
void with_vecs(int D, F &&f) {
  if (D <= 2048) f(std::integral_constant<int, 1>{});
  else if (D <= 4096) f(std::integral_constant<int, 2>{});
  else f(std::integral_constant<int, 4>{});
}

// post[n] * out + comb^T @ residual, f16 as the reference (its g5_hc_mix runs in
// block_out's dtype): each thread two adjacent d of one position, every n.
__global__ __launch_bounds__(256) void k_hc_mix(const uint16_t *__restrict__ bout, const float *__restrict__ post,
                                                const float *__restrict__ comb, const uint16_t *__restrict__ res,
                                                int64_t P, int N, int D, uint16_t *__restrict__ out) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int half_d = D / 2;
  if (g >= P * half_d) return;
  const int64_t p = g / half_d;
  const int d = (int)(g % half_d) * 2;
  const uint32_t b = *reinterpret_cast<const uint32_t *>(bout + p * D + d);
  uint32_t rv[exl3m::kHcMixMax];
  exl3m::hc_mix_res(res + p * N * D + d, D, N, rv);
  exl3m::hc_mix_pair(post + p * N, comb + p * N * N, rv, D, N, h2f(b & 0xffff), h2f(b >> 16),
                     out + p * N * D + d);
}

}  // namespace

namespace exl3h {

exl3_status check_hc(const exl3_hc_site *hc, int D) {
  if (!hc || !hc->fn || !hc->base || !hc->scale) return fail(EXL3_ERR_INVALID, "null hyper-connection site");
  if (hc->mult < 1 || hc->mult > kHcMaxN)
    return fail(EXL3_ERR_UNSUPPORTED, "hc_mult must be 1..8");
  if (hc->sinkhorn_iters < 1) return fail(EXL3_ERR_INVALID, "hc_sinkhorn_iters must be >= 1");
  if (D <= 0 || D > kHcMaxD || D % 2 || ((int64_t)hc->mult * D) % kHcChunk)
    return fail(EXL3_ERR_UNSUPPORTED, "hidden size must be even, at most 8192, and N*hidden a multiple of 64");
  return EXL3_OK;
}

// One partial per chunk: more than the groups' that calls of few positions write. Callers' sizes
// (and which calls a given workspace is refused for) stay as they were with a partial per chunk.
size_t hc_part_bytes(int N, int D, int64_t P) {
  return align_up((size_t)P * ((size_t)N * D / kHcChunk) * hc_vals(N) * 4, 256);
}

template <int kN, int NT>
static void hc_proj_go(bool many, const uint16_t *streams, int64_t P, int ND, int W, const float *fn, float *part,
                       int n_slices, hipStream_t st) {
  // (5 tiles of projections: one row tile per wave, within the registers of two waves a SIMD)
  constexpr int RT = NT <= 3 ? 2 : 1;
  const unsigned tiles = (unsigned)((P + kHcRows - 1) / kHcRows);
  if (many)
    k_hc_proj<kN, NT, RT, kHcFan><<<dim3((unsigned)n_slices, (unsigned)((P + kHcRows * RT - 1) / (kHcRows * RT))),
                                    64 * kHcWaves, 0, st>>>(streams, P, ND, W, fn, part);
  else if (NT > 2 && (int64_t)n_slices * tiles <= kHcSplitGroups)
    k_hc_proj<kN, 1, 1, 1><<<dim3((unsigned)n_slices, tiles, (unsigned)NT), 64 * kHcWaves, 0, st>>>(streams, P, ND, W,
                                                                                                fn, part);
  else
    k_hc_proj<kN, NT, 1, 1><<<dim3((unsigned)n_slices, tiles), 64 * kHcWaves, 0, st>>>(streams, P, ND, W, fn, part);
}

template <int kN>
static void hc_prepare_go(const exl3_hc_site *hc, const uint16_t *streams, int64_t P, int D,
                          const uint16_t *norm_w, float norm_eps, uint16_t *out, float *post, float *comb,
                          float *part, hipStream_t st) {
  const int N = hc->mult, W = (2 + N) * N, ND = N * D;
  const bool many = P >= kHcManyRows;
  const int n_slices = hc_slices(ND, many ? kHcFan * kHcFan : kHcFan);
  // tiles of 16 projections: up to 2 for 1..4 streams (W <= 24), 3..5 for 5..8 (35..80)
  constexpr int kT = kN <= kHcNarrowN ? 1 : 3;
  switch ((W + 15) / 16 - kT) {
    case 0: hc_proj_go<kN, kT>(many, streams, P, ND, W, hc->fn, part, n_slices, st); break;
    case 1: hc_proj_go<kN, kT + 1>(many, streams, P, ND, W, hc->fn, part, n_slices, st); break;
    default:
      if constexpr (kN > kHcNarrowN) hc_proj_go<kN, kT + 2>(many, streams, P, ND, W, hc->fn, part, n_slices, st);
  }
  const int64_t comb_blocks = many ? (P + HcShape<kN>::kPos - 1) / HcShape<kN>::kPos : P;
  with_vecs(D, [&](auto v) {
    k_hc_finalize<kN, decltype(v)::value><<<(unsigned)(comb_blocks + P), 256, 0, st>>>(
        streams, P, N, D, W, n_slices, many ? 1 : kHcFan, (int)comb_blocks, part, hc->base, hc->scale,
        hc->sinkhorn_iters, hc->eps, norm_w, norm_eps, out, post, comb);
  });
}

exl3_status launch_hc_prepare(const exl3_hc_site *hc, const uint16_t *streams, int64_t P, int D,
                              const uint16_t *norm_w, float norm_eps, uint16_t *out, float *post,
                              float *comb, float *part, hipStream_t st) {
  if (P == 0) return EXL3_OK;
  const bool narrow = hc->mult <= kHcNarrowN;
  // the positions of one call: 65,535 times 8, times 3 with more than 4 streams (a limit of the
  // call; the launches' grids take more)
  const int rows = narrow ? 8 : 3;
  if ((P + rows - 1) / rows > 65535) return fail(EXL3_ERR_UNSUPPORTED, "too many positions in one call");
  if (narrow)
    hc_prepare_go<kHcNarrowN>(hc, streams, P, D, norm_w, norm_eps, out, post, comb, part, st);
  else
    hc_prepare_go<kHcMaxN>(hc, streams, P, D, norm_w, norm_eps, out, post, comb, part, st);
  EXL3_LAUNCHED("k_hc_proj / k_hc_finalize");
  return EXL3_OK;
}

}  // namespace exl3h

using namespace exl3h;

extern "C" {

size_t exl3_hc_workspace_size(int32_t mult, int32_t hidden, int64_t P) {
  if (mult < 1 || mult > kHcMaxN || hidden <= 0 || P < 0 || ((int64_t)mult * hidden) % kHcChunk) return 0;
  return hc_part_bytes(mult, hidden, P);
}

exl3_status exl3_hc_prepare(const exl3_hc_site *hc, const uint16_t *streams, int64_t P, int32_t hidden,
                            const uint16_t *norm_w, float norm_eps, uint16_t *out, float *post, float *comb,
                            void *workspace, size_t workspace_bytes, exl3_stream_t stream) {
  exl3_status rc = check_hc(hc, hidden);
  if (rc) return rc;
  if (P < 0 || P > ((int64_t)1 << 31)) return fail(EXL3_ERR_INVALID, "exl3_hc_prepare: bad row count");
  if (P == 0) return EXL3_OK;
  if (!streams || !out || !post || !comb) return fail(EXL3_ERR_INVALID, "exl3_hc_prepare: null argument");
  const size_t need = hc_part_bytes(hc->mult, hidden, P);
  if (!workspace || workspace_bytes < need)
    return fail(EXL3_ERR_WORKSPACE, "exl3_hc_prepare: workspace too small: need " + std::to_string(need) + " bytes");
  if (reinterpret_cast<uintptr_t>(workspace) % 256)
    return fail(EXL3_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  if (reinterpret_cast<uintptr_t>(streams) % 8 || reinterpret_cast<uintptr_t>(hc->fn) % 16 ||
      (reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(norm_w)) % 4)
    return fail(EXL3_ERR_INVALID, "streams must be 8-byte, fn 16-byte, out and norm_w 4-byte aligned");
  return launch_hc_prepare(hc, streams, P, hidden, norm_w, norm_eps, out, post, comb, (float *)workspace,
                           stream_of(stream));
}

exl3_status exl3_rms_norm(const uint16_t *x, int64_t P, int32_t hidden, const uint16_t *w, float eps, uint16_t *y,
                          exl3_stream_t stream) {
  if (P < 0 || P > ((int64_t)1 << 31) || hidden <= 0 || hidden > kHcMaxD || hidden % 2)
    return fail(EXL3_ERR_INVALID, "exl3_rms_norm: bad shape (hidden even, at most 8192)");
  if (P == 0) return EXL3_OK;
  if (!x || !w || !y) return fail(EXL3_ERR_INVALID, "exl3_rms_norm: null argument");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) % 4)
    return fail(EXL3_ERR_INVALID, "exl3_rms_norm: x, w and y must be 4-byte aligned");
  with_vecs(hidden, [&](auto v) {
    k_rms_norm<decltype(v)::value><<<(unsigned)P, 256, 0, stream_of(stream)>>>(x, hidden, w, eps, y);
  });
  EXL3_LAUNCHED("k_rms_norm");
  return EXL3_OK;
}

exl3_status exl3_hc_mix(const uint16_t *block_out, const float *post, const float *comb, const uint16_t *residual,
                        int64_t P, int32_t mult, int32_t hidden, uint16_t *out, exl3_stream_t stream) {
  if (P < 0 || mult < 1 || mult > kHcMaxN || hidden <= 0 || hidden % 2)
    return fail(EXL3_ERR_INVALID, "exl3_hc_mix: bad shape (hc_mult 1..8, even hidden)");
  if (P == 0) return EXL3_OK;
  if (!block_out || !post || !comb || !residual || !out) return fail(EXL3_ERR_INVALID, "exl3_hc_mix: null argument");
  if ((reinterpret_cast<uintptr_t>(block_out) | reinterpret_cast<uintptr_t>(residual) |
       reinterpret_cast<uintptr_t>(out)) % 4)
    return fail(EXL3_ERR_INVALID, "exl3_hc_mix: block_out, residual and out must be 4-byte aligned");
  if (P > ((int64_t)1 << 40) / hidden) return fail(EXL3_ERR_UNSUPPORTED, "exl3_hc_mix: too large");
  if (overlaps(residual, out, (size_t)P * mult * hidden * 2))
    return fail(EXL3_ERR_INVALID, "exl3_hc_mix: out must not overlap residual");
  const int64_t threads = P * (hidden / 2);
  if (threads == 0) return EXL3_OK;
  k_hc_mix<<<(unsigned)((threads + 255) / 256), 256, 0, stream_of(stream)>>>(block_out, post, comb, residual, P,
                                                                             mult, hidden, out);
  EXL3_LAUNCHED("k_hc_mix");
  return EXL3_OK;
}

}  // extern "C"
