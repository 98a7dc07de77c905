// Row softmax device code: the element math and the row bodies of the two asc2
// softmax kernels
//   test_softmax.py:16-27        grid-stride rows, one [1, tile_size] tile per row
//   test_softmax_fused.py:16-24  contiguous row blocks through asc2.softmax
// (python/test/asc2/kernels/).  Both reduce to: for each covered row r,
// out[r, :L] = exp(x - max) / sum(exp(x - max)) over the row's first L columns
// (row stride S).  Shared by the library (softmax.hip, launched through
// asc_softmax_*) and the standalone gfx950 code object (co/asc2_softmax.hip,
// loaded with hipModuleLoad by the asc2 launch path), so both launch paths run
// the same instructions.
//
// Every body takes the same six arguments,
//   (x, out, rows, stride, len, flag)
// where flag is "rows start 16-byte aligned" for the fp32 bodies (which load and
// store at element alignment and do not need it), "rows are made of aligned
// 16-byte vectors" for the f16 bodies and the pad count (tile - num_cols) for the
// padded bodies.
//
// HBM-bound (one read + one write of every element).  Rows up to 49152 fp32 or 65529
// fp16 columns stay in registers: 16 lanes, a wave or a workgroup per row, by its
// length and the number of rows (asc_softmax_dispatch picks the body).  Max,
// min and sum reduce in-thread, then across the wave with DPP and permlane
// swaps (no LDS round trips), then across waves through LDS.  x - max is
// rounded to fp32 as in the reference (test_softmax.py:22-24); exp of it is
// accurate to ~2 ulp (the row's min picks a shorter exp when no result can fall
// below 2^-126) and the normalisation multiplies by one correctly rounded
// reciprocal per row, which stays within 2 ulp of the reference's true division
// (DivL2, lib/Conversion/LowerToAsc/LowerArithBinary.cpp:116).
#pragma once

#include <math.h>

#include "common.h"
#include "rows.h"

namespace asc {
namespace softmax {

using asc::rows::f32x4;
using asc::rows::load_row;
using asc::rows::load_vec;
using asc::rows::RowView;
using asc::rows::store_row;
using asc::rows::store_vec;

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// softmax rows are padded with -inf (no effect on max, sum or the exp path)
constexpr float kPad = -INFINITY;

constexpr float kL2E = 1.44269504088896340736f;   // log2(e) rounded to fp32
constexpr float kL2ELo = 1.925963033500011e-08f;  // log2(e) - kL2E
constexpr float kLn2 = 0.69314718055994530942f;
constexpr float kMinNormalLog2 = -126.0f;

// Normalises the row in registers and stores it.
template <int N, int kStride>
__device__ __forceinline__ void store_scaled(float4 (&v)[N], float* row, int q0, int len, float rs) {
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = make_float4(v[j].x * rs, v[j].y * rs, v[j].z * rs, v[j].w * rs);
  store_row<N, kStride>(v, row, q0, len);
}

// exp(y) for finite y <= 0 with y*log2(e) >= -126 (the caller checks the row's
// range), within ~2 ulp: t = y*log2(e) rounded, v_exp_f32 of t, and a
// first-order correction by the rounding residual, taken from a two-term split
// of log2(e) (Cody-Waite).
__device__ __forceinline__ float exp_plain(float y) {
  const float t = y * kL2E;
  const float err = fmaf(y, kL2ELo, fmaf(y, kL2E, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, err * kLn2, e);
}

// exp(y) for any y <= 0 (-inf gives 0, NaN stays NaN).  v_exp_f32 flushes
// results below 2^-126, so those are evaluated 64 octaves up (t + 64 is exact
// for t <= -126) and scaled back by an exact power of two, which rounds once
// into the denormal range.
__device__ __forceinline__ float exp_nonpos(float y) {
  const float t = y * kL2E;
  const float yc = fmaxf(y, -104.0f);  // keeps the residual finite for y = -inf
  const float err = fmaf(yc, kL2ELo, fmaf(yc, kL2E, -(yc * kL2E)));
  const bool tiny = t < kMinNormalLog2;
  const float e = __builtin_amdgcn_exp2f(tiny ? t + 64.0f : t);
  const float r = fmaf(e, err * kLn2, e);
  return tiny ? r * 0x1p-64f : r;
}

// True when every exp(x - m) of a row with maximum m and minimum mn is a
// normal number reached by exp_plain: RN(RN(mn - m) * log2 e) >= -126 bounds
// RN(RN(x - m) * log2 e) for every x of the row (rounding is monotonic).
// mn = -inf (a -inf element or padding) selects the general path.
__device__ __forceinline__ bool plain_range(float m, float mn) { return (mn - m) * kL2E >= kMinNormalLog2; }

// exp(v - m) per lane of a vector
template <bool kPlain>
__device__ __forceinline__ float4 exp_shift(float4 v, float m) {
  float4 r;
  if constexpr (kPlain) {
    r.x = exp_plain(v.x - m);
    r.y = exp_plain(v.y - m);
    r.z = exp_plain(v.z - m);
    r.w = exp_plain(v.w - m);
  } else {
    r.x = exp_nonpos(v.x - m);
    r.y = exp_nonpos(v.y - m);
    r.z = exp_nonpos(v.z - m);
    r.w = exp_nonpos(v.w - m);
  }
  return r;
}

__device__ __forceinline__ float max4(float4 v) { return fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)); }
__device__ __forceinline__ float min4(float4 v) { return fminf(fminf(v.x, v.y), fminf(v.z, v.w)); }

// Replaces the vectors of one row by exp(v - m) and returns their sum.  One
// vector at a time (scheduling fence): with many waves per SIMD resident,
// overlapping the exps of several vectors buys nothing and its temporaries
// would cost occupancy.  Long shares are summed in several chains (fewer roundings in a row).
template <int N>
__device__ __forceinline__ float exp_row(float4 (&v)[N], float m, float mn) {
  constexpr int kChains = N > 8 ? 4 : N > 4 ? 2 : 1;
  float s[kChains] = {};
  if (plain_range(m, mn)) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      v[j] = exp_shift<true>(v[j], m);
      s[j % kChains] += (v[j].x + v[j].y) + (v[j].z + v[j].w);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      v[j] = exp_shift<false>(v[j], m);
      s[j % kChains] += (v[j].x + v[j].y) + (v[j].z + v[j].w);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (kChains == 4) return (s[0] + s[1]) + (s[2] + s[3]);
  if constexpr (kChains == 2) return s[0] + s[1];
  return s[0];
}

__device__ __forceinline__ RowView row_view(const void* x, void* out, int64_t rows, int64_t stride, int32_t len) {
  return RowView{static_cast<const float*>(x), static_cast<float*>(out), rows, stride, len};
}

// One wave per row; each lane holds VPL float4 vectors of each of kRows rows
// (all rows' loads are issued before any reduction, so more bytes are in flight).
// 256-thread blocks, four waves: block b covers rows [8b, 8b + 8) for kRows = 2.
template <int VPL, int kRows>
__device__ __forceinline__ void wave_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                          int32_t) {
  const RowView p = row_view(x, out, rows, stride, len);
  const int lane = threadIdx.x & 63;
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * kRows;
  float4 v[kRows][VPL];
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    if (r0 + k >= p.rows) continue;
    load_row<VPL, 64>(v[k], p.x + (r0 + k) * p.stride, lane, p.len, kPad);
  }
#pragma unroll
  for (int k = 0; k < kRows; ++k) {
    if (r0 + k >= p.rows) continue;
    float m = -INFINITY, mn = INFINITY;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      m = fmaxf(m, max4(v[k][j]));
      mn = fminf(mn, min4(v[k][j]));
    }
    m = asc::wave_max(m);
    mn = asc::wave_min(mn);
    const float rs = 1.0f / asc::wave_sum(exp_row(v[k], m, mn));
    store_scaled<VPL, 64>(v[k], p.out + (r0 + k) * p.stride, lane, p.len, rs);
  }
}

// The sum of the waves' sums, kExact in fp64: this rounding error is the same in every result of a
// row (relative error against fp64: 2000x8193, 4 waves, 7.39e-8 with an fp32 chain, 7.03e-8 with
// fp64; 300x100003, 16 waves, 9.9e-8 and 8.6e-8).
template <int kWaves, bool kExact>
__device__ __forceinline__ float sum_waves(const float (&red)[kWaves]) {
  if constexpr (kExact) {
    double sum = red[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += red[w];
    return static_cast<float>(sum);
  }
  float sum = red[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) sum += red[w];
  return sum;
}

// One kThreads-thread block per row (block b is row b); each thread holds VPT
// float4 vectors.  The cross-wave max/min and sum go through LDS, one barrier each.
template <int VPT, int kThreads>
__device__ __forceinline__ void block_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                           int32_t) {
  const RowView p = row_view(x, out, rows, stride, len);
  constexpr int kWaves = kThreads / 64;
  __shared__ float red[3][kWaves];  // max, min, sum per wave
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x;
  float4 v[VPT];
  load_row<VPT, kThreads>(v, p.x + r * p.stride, t, p.len, kPad);
  float m = -INFINITY, mn = INFINITY;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    m = fmaxf(m, max4(v[j]));
    mn = fminf(mn, min4(v[j]));
  }
  m = asc::wave_max(m);
  mn = asc::wave_min(mn);
  if ((t & 63) == 0) {
    red[0][t >> 6] = m;
    red[1][t >> 6] = mn;
  }
  __syncthreads();
  m = red[0][0];
  mn = red[1][0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    m = fmaxf(m, red[0][w]);
    mn = fminf(mn, red[1][w]);
  }
  const float s = asc::wave_sum(exp_row(v, m, mn));
  if ((t & 63) == 0) red[2][t >> 6] = s;
  __syncthreads();
  store_scaled<VPT, kThreads>(v, p.out + r * p.stride, t, p.len, 1.0f / sum_waves<kWaves, (VPT > 8 || kWaves > 8)>(red[2]));
}

// Maximum and sum over a group of kLanes threads: 16, 64 or the whole workgroup.
template <int kLanes>
__device__ __forceinline__ float group_max(float v, float* red) {
  if constexpr (kLanes == 16) {
    v = fmaxf(v, asc::dpp_mov<asc::kDppQuadXor1>(v));
    v = fmaxf(v, asc::dpp_mov<asc::kDppQuadXor2>(v));
    v = fmaxf(v, asc::dpp_mov<asc::kDppRowHalfMirror>(v));
    return fmaxf(v, asc::dpp_mov<asc::kDppRowMirror>(v));
  }
  v = asc::wave_max(v);
  if constexpr (kLanes == 64) return v;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int w = 1; w < kLanes / 64; ++w) v = fmaxf(v, red[w]);
  return v;
}
template <int kLanes>
__device__ __forceinline__ float group_sum(float v, float* red) {
  if constexpr (kLanes == 16) {
    v += asc::dpp_mov<asc::kDppQuadXor1>(v);
    v += asc::dpp_mov<asc::kDppQuadXor2>(v);
    v += asc::dpp_mov<asc::kDppRowHalfMirror>(v);
    return v + asc::dpp_mov<asc::kDppRowMirror>(v);
  }
  v = asc::wave_sum(v);
  if constexpr (kLanes == 64) return v;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int w = 1; w < kLanes / 64; ++w) v += red[w];
  return v;
}

// The value of another lane of the 16, as asc::dpp_mov.
template <int kCtrl>
__device__ __forceinline__ double dpp_mov64(double v) {
  const u32x2_t b = __builtin_bit_cast(u32x2_t, v);
  const u32x2_t r = {__float_as_uint(asc::dpp_mov<kCtrl>(__uint_as_float(b[0]))),
                     __float_as_uint(asc::dpp_mov<kCtrl>(__uint_as_float(b[1])))};
  return __builtin_bit_cast(double, r);
}

// Sum over 16 lanes in fp64: with up to eight vectors per lane in a chain, fp32 rounded the sum
// more than a wave per row did (relative error against fp64, values within 0.1 of each other:
// 192 columns 5.9e-8 with a wave, 6.2e-8 in fp32, 5.2e-8 here; 384: 6.0e-8, 6.3e-8, 5.3e-8); the
// time is the same (30000x384: 15.6 us).
__device__ __forceinline__ double sum16(double v) {
  v += dpp_mov64<asc::kDppQuadXor1>(v);
  v += dpp_mov64<asc::kDppQuadXor2>(v);
  v += dpp_mov64<asc::kDppRowHalfMirror>(v);
  return v + dpp_mov64<asc::kDppRowMirror>(v);
}

// Short rows, 16 lanes per row and VPT vectors per lane: 256-thread block b covers rows
// [16b, 16b + 16).  Bound by how many loads and reductions a wave issues per row: four rows per
// wave share each of them, and fewer lanes lie past a short row's end than with a wave per row
// (wave_1x2/wave_2x2 before, here; us: 200000x64 52.3, 20.4; 100000x67 29.5, 15.0; 30000x256
// 13.8, 12.1; 30000x333 25.6, 19.2).
template <int VPT>
__device__ __forceinline__ void short_rows(const void* x, void* out, int64_t rows, int64_t stride, int32_t len) {
  const RowView p = row_view(x, out, rows, stride, len);
  const int t = threadIdx.x & 15;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x >> 4);
  if (r >= p.rows) return;
  float4 v[VPT];
  load_row<VPT, 16>(v, p.x + r * p.stride, t, p.len, kPad);
  float m = -INFINITY, mn = INFINITY;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    m = fmaxf(m, max4(v[j]));
    mn = fminf(mn, min4(v[j]));
  }
  m = group_max<16>(m, nullptr);
  mn = -group_max<16>(-mn, nullptr);
  const float rs = 1.0f / static_cast<float>(sum16(exp_row(v, m, mn)));
  store_scaled<VPT, 16>(v, p.out + r * p.stride, t, p.len, rs);
}

__device__ __forceinline__ void short_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                           int32_t) {
  if (len <= 64) short_rows<1>(x, out, rows, stride, len);
  else if (len <= 128) short_rows<2>(x, out, rows, stride, len);
  else if (len <= 192) short_rows<3>(x, out, rows, stride, len);
  else if (len <= 256) short_rows<4>(x, out, rows, stride, len);
  else if (len <= 384) short_rows<6>(x, out, rows, stride, len);
  else short_rows<8>(x, out, rows, stride, len);
}

// exp(y) for any y <= 0, results below 2^-126 flushed to 0 (as terms of a sum whose largest
// is 1, or on the way to fp16, they round away): -inf gives 0, NaN stays NaN.
__device__ __forceinline__ float exp_flush(float y) {
  const float t = y * kL2E;
  const float err = fmaf(y, kL2ELo, fmaf(y, kL2E, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return t < kMinNormalLog2 ? 0.0f : fmaf(e, err * kLn2, e);
}

// A running maximum and the sum of exp(x - maximum) over a thread's share of a row.  -inf
// elements (and the -inf maximum of a share that has no others) add 0, a NaN makes the sum NaN.
struct OnlineSum {
  float m = -INFINITY, s = 0.0f;
  // Moves the maximum up to at least `to`.
  __device__ __forceinline__ void raise(float to) {
    const float m1 = fmaxf(m, to);
    if (m1 > m) {
      s *= exp_flush(m - m1);  // m = -inf: s is 0 or NaN
      m = m1;
    }
  }
  __device__ __forceinline__ float term(float x) const { return exp_flush(x - (m == -INFINITY ? 0.0f : m)); }
};

// Rows beyond the registers, one kThreads-thread workgroup per row, read twice: once for the
// maximum and the sum of each thread's share (eight vectors, one rescaling at a time), once
// to write the result.  HBM-bound (640x100003: 337 us with separate maximum and sum passes,
// 146 us with 1024 threads, 12 B per element at 5.3 TB/s).
template <int kThreads>
__device__ __forceinline__ void two_pass_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len) {
  const RowView p = row_view(x, out, rows, stride, len);
  constexpr int kWaves = kThreads / 64;
  __shared__ float red[3][kWaves];
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x;
  const float* row = p.x + r * p.stride;
  const int nvec = p.len / 4 + (p.len % 4 != 0);
  OnlineSum acc;
  float mn = INFINITY;
  constexpr int kChunk = 8;
  for (int q = t; q < nvec; q += kThreads * kChunk) {
    float4 v[kChunk];
    if (q + kThreads * (kChunk - 1) < p.len / 4) {
#pragma unroll
      for (int u = 0; u < kChunk; ++u) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(row + 4 * (q + kThreads * u));
        v[u] = make_float4(w.x, w.y, w.z, w.w);
      }
    } else {
#pragma unroll
      for (int u = 0; u < kChunk; ++u) {
        // a vector past the row is not asked for: its first element may not fit an int
        v[u] = make_float4(kPad, kPad, kPad, kPad);
        if (q + kThreads * u < nvec) v[u] = load_vec(row, q + kThreads * u, p.len, kPad);
      }
    }
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < kChunk; ++u) {
      m = fmaxf(m, max4(v[u]));
      mn = fminf(mn, min4(v[u]));
    }
    acc.raise(m);
#pragma unroll
    for (int u = 0; u < kChunk; ++u) {
      acc.s += (acc.term(v[u].x) + acc.term(v[u].y)) + (acc.term(v[u].z) + acc.term(v[u].w));
    }
  }
  float m = asc::wave_max(acc.m);
  mn = asc::wave_min(mn);
  if ((t & 63) == 0) {
    red[0][t >> 6] = m;
    red[1][t >> 6] = mn;
  }
  __syncthreads();
  m = red[0][0];
  mn = red[1][0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    m = fmaxf(m, red[0][w]);
    mn = fminf(mn, red[1][w]);
  }
  acc.raise(m);
  const float s = asc::wave_sum(acc.s);
  if ((t & 63) == 0) red[2][t >> 6] = s;
  __syncthreads();
  const float rs = 1.0f / sum_waves<kWaves, true>(red[2]);
  float* orow = p.out + r * p.stride;
#pragma unroll 4
  for (int q = t; q < nvec; q += kThreads) {
    float4 v[1] = {load_vec(row, q, p.len, kPad)};
    exp_row(v, m, mn);
    store_vec(orow, q, p.len, make_float4(v[0].x * rs, v[0].y * rs, v[0].z * rs, v[0].w * rs));
  }
}

// Rows longer than the 8192 columns of block_8x256: 256 threads per row, registers up to 16384
// columns (16 vectors per thread; 32 would leave one wave per SIMD).
__device__ __forceinline__ void long_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                          int32_t) {
  if (len <= 16 * 1024) block_body<16, 256>(x, out, rows, stride, len, 0);
  else two_pass_body<256>(x, out, rows, stride, len);
}

// Rows past 16384 columns, 1024 threads per row: the registers of sixteen waves hold up to
// 49152 columns, so x is read once (16 vectors per thread would spill), and few rows keep more
// loads in flight.  256 threads in two passes, here (us): 1500x20001 78.6, 69.2; 256x50000 51.5,
// 31.6; 8x100003 56.1, 24.7.  Up to 16384 columns, where 256 threads hold the row, they are the
// better: 1500x12001 31.6, 42.0 with 1024.
__device__ __forceinline__ void wide_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                          int32_t) {
  if (len <= 32 * 1024) block_body<8, 1024>(x, out, rows, stride, len, 0);
  else if (len <= 48 * 1024) block_body<12, 1024>(x, out, rows, stride, len, 0);
  else two_pass_body<1024>(x, out, rows, stride, len);
}

// ---- float16 rows (asc2.softmax on an f16 tile, python/asc/language/tile/unary_ops.py:213-222;
// python/test/asc2/operations/test_softmax.py).  fp32 statistics: x - max rounded to fp32, exp
// to about 2 ulp, one reciprocal of the sum, then one RNE rounding of each output to fp16.
// A row belongs to 16 lanes (up to 505 columns), a wave (up to 4089), a workgroup of 256
// threads (up to 16377) or one of 1024, and stays in registers as fp32, up to 64 values per
// thread, so x is read once; past 65529 columns it is read twice.  A row starts on any half,
// and 16-byte accesses at odd halves run at half rate, so vectors are aligned in memory, not
// to the row: vector q holds the row's elements 8q - h .. 8q - h + 7, h the halves between the
// row and the aligned address before it, and elements outside the row become -inf.  HBM-bound
// (4 B per element); a workgroup per row and separate passes for maximum, sum and result
// before, here (us): 3000x10007 87.6, 25.9; 4096x4096 23.6, 16.8; 100000x64 117, 12.4;
// 30000x1000 62, 25; 11926x2314 78, 25; 2000x32000 101, 63; 640x100003 385, 95.
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ float half_at(const uint16_t* p, int i) {
  return static_cast<float>(__builtin_bit_cast(_Float16, p[i]));
}
__device__ __forceinline__ uint16_t to_half(float v) {
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
}

constexpr uint32_t kHalfNegInf = 0xFC00u;

__device__ __forceinline__ void halves8(u32x4_t v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v[i] & 0xffffu)));
    f[2 * i + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v[i] >> 16)));
  }
}

// A row as vectors of eight halves.
struct HalfRow {
  const uint16_t* x;  // the aligned address at or before the row's first element
  uint16_t* out;      // as far before the output row's first element
  int h, end;         // the row is elements [h, end) from x
  int last;           // no vector starts after this element
  __device__ __forceinline__ HalfRow(const uint16_t* xs, uint16_t* outs, int64_t r, int64_t rows, int64_t stride,
                                     int32_t len) {
    const uint16_t* row = xs + r * stride;
    h = static_cast<int>(reinterpret_cast<uintptr_t>(row) & 15) >> 1;
    const bool inside = (h == 0 || r * stride >= 8) && (((h + (len & 7)) & 7) == 0 || (rows - 1 - r) * stride >= 8) &&
                        len <= INT32_MAX - 16;
    // Where an aligned vector would leave the tensor (its first or last row), or its end an int,
    // vectors start at the row, and the last one is moved back over elements that the one before
    // it holds.
    if (!inside) h = 0;
    x = row - h;
    out = outs + r * stride - h;
    end = h + len;
    last = inside ? end : len - 8;
  }
  __device__ __forceinline__ int vectors() const { return end / 8 + (end % 8 != 0); }
  __device__ __forceinline__ bool tiny() const { return last < 0; }  // less than a vector to read
  __device__ __forceinline__ int first(int q) const { return min(8 * q, last); }

  // Vector q < vectors(), -inf in place of elements outside the row or held by vector q - 1.
  __device__ __forceinline__ u32x4_t load(int q) const {
    const int at = first(q);
    u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(x + at));
    const int lo = max(h, 8 * q) - at, hi = end - at;  // elements [lo, hi) of the vector are taken
    if (lo > 0 || hi < 8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (2 * i < lo || 2 * i >= hi) v[i] = (v[i] & 0xffff0000u) | kHalfNegInf;
        if (2 * i + 1 < lo || 2 * i + 1 >= hi) v[i] = (v[i] & 0xffffu) | (kHalfNegInf << 16);
      }
    }
    return v;
  }
  __device__ __forceinline__ void store(int q, const float (&f)[8], float scale) const {
    const int at = first(q);
    const int lo = max(h, 8 * q) - at, hi = end - at;
    uint16_t v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = to_half(f[i] * scale);
    uint16_t* o = out + at;
    if (lo <= 0 && hi >= 8) {
      u32x4_any w;
      __builtin_memcpy(&w, v, 16);
      __builtin_nontemporal_store(w, reinterpret_cast<u32x4_any*>(o));
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i >= lo && i < hi) o[i] = v[i];
    }
  }
};

__device__ __forceinline__ float max8(const float (&f)[8]) {
  return fmaxf(fmaxf(fmaxf(f[0], f[1]), fmaxf(f[2], f[3])), fmaxf(fmaxf(f[4], f[5]), fmaxf(f[6], f[7])));
}
__device__ __forceinline__ float sum8(const float (&f)[8]) {
  return ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
}

// A first or last row of fewer than eight halves, one per lane.
template <int kLanes>
__device__ __forceinline__ void f16_tiny_row(const uint16_t* row, uint16_t* out, int32_t len, int t, float (*red)[16]) {
  const float v = t < len ? half_at(row, t) : -INFINITY;
  const float e = exp_flush(v - group_max<kLanes>(v, red[0]));
  const float rs = 1.0f / group_sum<kLanes>(e, red[1]);
  if (t < len) out[t] = to_half(e * rs);
}

// Rows of up to 8 * VPT * kLanes - 7 halves, one per group of kLanes of the workgroup's threads.
template <int VPT, int kLanes, int kThreads>
__device__ __forceinline__ void f16_rows(const uint16_t* x, uint16_t* out, int64_t rows, int64_t stride, int32_t len,
                                         float (*red)[16]) {
  constexpr int kGroups = kThreads / kLanes;
  const int t = threadIdx.x % kLanes;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * kGroups + threadIdx.x / kLanes; r < rows;
       r += static_cast<int64_t>(gridDim.x) * kGroups) {
    const HalfRow row(x, out, r, rows, stride, len);
    if (row.tiny()) {
      f16_tiny_row<kLanes>(x + r * stride, out + r * stride, len, t, red);
      continue;
    }
    const int nvec = row.vectors();
    u32x4_t raw[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      constexpr uint32_t kNone = kHalfNegInf | kHalfNegInf << 16;
      raw[j] = u32x4_t{kNone, kNone, kNone, kNone};
      if (t + kLanes * j < nvec) raw[j] = row.load(t + kLanes * j);
    }
    float f[VPT][8];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      halves8(raw[j], f[j]);
      m = fmaxf(m, max8(f[j]));
    }
    m = group_max<kLanes>(m, red[0]);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
#pragma unroll
      for (int i = 0; i < 8; ++i) f[j][i] = exp_flush(f[j][i] - m);
      s += sum8(f[j]);
    }
    const float rs = 1.0f / group_sum<kLanes>(s, red[1]);
#pragma unroll
    for (int j = 0; j < VPT; ++j)
      if (t + kLanes * j < nvec) row.store(t + kLanes * j, f[j], rs);
  }
}

// Few rows that are not made of aligned vectors, element by element: kPer per lane, a row per
// group of kLanes of the workgroup's threads.  With few rows the latency of one counts, and the
// masks of a vector at a row's ends cost more of it than loads of an element each (an element per
// thread before, vectors, here; us): 16x122 2.3, 2.7, 2.0; 128x506 2.9, 3.3, 2.2; 512x1017 3.8,
// 3.8, 2.6; 1000x122 2.9, 2.9, 2.1; 1000x1017 4.7, 4.0, 3.0.
template <int kPer, int kLanes>
__device__ __forceinline__ void f16_element_rows(const uint16_t* x, uint16_t* out, int64_t rows, int64_t stride,
                                                 int32_t len, float (*red)[16]) {
  constexpr int kGroups = 256 / kLanes;
  const int t = threadIdx.x % kLanes;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * kGroups + threadIdx.x / kLanes; r < rows;
       r += static_cast<int64_t>(gridDim.x) * kGroups) {
    float f[kPer];
    float m = -INFINITY, s = 0.0f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      f[j] = t + kLanes * j < len ? half_at(x + r * stride, t + kLanes * j) : -INFINITY;
      m = fmaxf(m, f[j]);
    }
    m = group_max<kLanes>(m, red[0]);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      f[j] = exp_flush(f[j] - m);
      s += f[j];
    }
    const float rs = 1.0f / group_sum<kLanes>(s, red[1]);
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if (t + kLanes * j < len) out[r * stride + t + kLanes * j] = to_half(f[j] * rs);
  }
}

// Longer rows, one per workgroup, in two passes.
template <int kThreads>
__device__ __forceinline__ void f16_long_rows(const uint16_t* x, uint16_t* out, int64_t rows, int64_t stride,
                                              int32_t len, float (*red)[16]) {
  const int t = threadIdx.x;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const HalfRow row(x, out, r, rows, stride, len);
    const int nvec = row.vectors();
    OnlineSum acc;
#pragma unroll 4
    for (int q = t; q < nvec; q += kThreads) {
      float f[8];
      halves8(row.load(q), f);
      acc.raise(max8(f));
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = acc.term(f[i]);
      acc.s += sum8(f);
    }
    const float m = group_max<kThreads>(acc.m, red[0]);
    acc.raise(m);
    const float rs = 1.0f / group_sum<kThreads>(acc.s, red[1]);
#pragma unroll 2
    for (int q = t; q < nvec; q += kThreads) {
      float f[8];
      halves8(row.load(q), f);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = exp_flush(f[i] - m);
      row.store(q, f, rs);
    }
  }
}

// Rows of len halves that a 256-thread workgroup of f16_body takes at once.  Fewer lanes per row
// leave fewer of them past its end and shorten the reductions (60000x333: 23 us with 16 lanes, 35
// with a wave per row; 11926x2314: 25 with a wave, 45 with a workgroup); with few rows the
// row's own latency counts and more lanes are better (300x333: 3.2 us with a wave, 4.1 with 16
// lanes, even at about 2000 rows; 1000x4000: 5.7 with a workgroup, 8x4000: 3.1, 4.7 with a wave,
// even at about 1000 rows).
constexpr bool f16_by_elements(int32_t len, int64_t rows, bool aligned) {
  return !aligned && len <= 1017 && rows <= 1024;
}
constexpr int32_t f16_rows_per_block(int32_t len, int64_t rows, bool aligned) {
  if (f16_by_elements(len, rows, aligned)) return len <= 256 ? 4 : 1;
  if (len <= 505) return len <= 121 || rows > 2048 ? 16 : 4;
  return len <= 1017 || (len <= 4089 && rows > 1024) ? 4 : 1;
}

// aligned: rows are made of 16-byte vectors at aligned addresses.
__device__ __forceinline__ void f16_body(const void* xv, void* outv, int64_t rows, int64_t stride, int32_t len,
                                         int32_t aligned) {
  __shared__ float red[2][16];
  const uint16_t* x = static_cast<const uint16_t*>(xv);
  uint16_t* out = static_cast<uint16_t*>(outv);
  if (f16_by_elements(len, rows, aligned != 0)) {
    if (len <= 64) return f16_element_rows<1, 64>(x, out, rows, stride, len, red);
    if (len <= 128) return f16_element_rows<2, 64>(x, out, rows, stride, len, red);
    if (len <= 256) return f16_element_rows<4, 64>(x, out, rows, stride, len, red);
    if (len <= 512) return f16_element_rows<2, 256>(x, out, rows, stride, len, red);
    if (len <= 768) return f16_element_rows<3, 256>(x, out, rows, stride, len, red);
    return f16_element_rows<4, 256>(x, out, rows, stride, len, red);
  }
  if (len <= 121) return f16_rows<1, 16, 256>(x, out, rows, stride, len, red);
  if (len <= 505 && rows <= 2048) return f16_rows<1, 64, 256>(x, out, rows, stride, len, red);
  if (len > 1017 && rows <= 1024) {
    if (len <= 2041) return f16_rows<1, 256, 256>(x, out, rows, stride, len, red);
    if (len <= 4089) return f16_rows<2, 256, 256>(x, out, rows, stride, len, red);
  }
  if (len <= 249) return f16_rows<2, 16, 256>(x, out, rows, stride, len, red);
  if (len <= 377) return f16_rows<3, 16, 256>(x, out, rows, stride, len, red);
  if (len <= 505) return f16_rows<4, 16, 256>(x, out, rows, stride, len, red);
  if (len <= 1017) return f16_rows<2, 64, 256>(x, out, rows, stride, len, red);
  if (len <= 1529) return f16_rows<3, 64, 256>(x, out, rows, stride, len, red);
  if (len <= 2041) return f16_rows<4, 64, 256>(x, out, rows, stride, len, red);
  if (len <= 3065) return f16_rows<6, 64, 256>(x, out, rows, stride, len, red);
  if (len <= 4089) return f16_rows<8, 64, 256>(x, out, rows, stride, len, red);
  if (len <= 6137) return f16_rows<3, 256, 256>(x, out, rows, stride, len, red);
  if (len <= 8185) return f16_rows<4, 256, 256>(x, out, rows, stride, len, red);
  if (len <= 10233) return f16_rows<5, 256, 256>(x, out, rows, stride, len, red);
  if (len <= 12281) return f16_rows<6, 256, 256>(x, out, rows, stride, len, red);
  if (len <= 16377) return f16_rows<8, 256, 256>(x, out, rows, stride, len, red);
  f16_long_rows<256>(x, out, rows, stride, len, red);
}

// 1024 threads per row, for rows past 16377 columns (registers up to 65529).
__device__ __forceinline__ void f16_wide_body(const void* xv, void* outv, int64_t rows, int64_t stride, int32_t len,
                                              int32_t) {
  __shared__ float red[2][16];
  const uint16_t* x = static_cast<const uint16_t*>(xv);
  uint16_t* out = static_cast<uint16_t*>(outv);
  if (len <= 32761) return f16_rows<4, 1024, 1024>(x, out, rows, stride, len, red);
  if (len <= 65529) return f16_rows<8, 1024, 1024>(x, out, rows, stride, len, red);
  f16_long_rows<1024>(x, out, rows, stride, len, red);
}

// ---- tiles wider than the row (test_softmax.py's softmax_kernel with tile_size >
// num_cols).  The reference's load right-pads the [1, tile] tile with the pad value 0
// (lib/Conversion/LowerToAsc/LowerAscTileDataTransfer.cpp:181-222) and its reductions
// count the whole tile (lib/Conversion/LowerToAsc/LowerAscTile.cpp:428-459), so each
// row's statistics include pad = tile - num_cols zeros:
//   m = max(max_j x_j, 0),  s = sum_j exp(x_j - m) + pad * exp(-m),  out_j = exp(x_j - m) / s.
// Its store then writes the whole tile from the row's start, spilling pad values
// into the next row, where they race with that row's own store whenever the two rows
// run on different blocks; here every row writes its own num_cols values only (what
// running the rows in order on one block leaves).  256-thread workgroups over rows
// b, b + gridDim.x, ..., three passes (rows are contiguous: stride = len = num_cols);
// not a tuned path.
template <bool kHalf>
__device__ __forceinline__ float padded_at(const void* row, int64_t c) {
  if constexpr (kHalf) return half_at(static_cast<const uint16_t*>(row), static_cast<int>(c));
  else return static_cast<const float*>(row)[c];
}

template <bool kHalf>
__device__ __forceinline__ void padded_body(const void* x, void* out, int64_t rows, int64_t stride, int32_t len,
                                            int32_t pad) {
  __shared__ float red[2][4];
  const int t = threadIdx.x;
  constexpr int64_t kES = kHalf ? 2 : 4;
  const int64_t cols = len;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const void* row = static_cast<const uint8_t*>(x) + r * stride * kES;
    float m = pad > 0 ? 0.0f : -INFINITY;  // the padding zeros take part in the maximum
    for (int64_t c = t; c < cols; c += 256) m = fmaxf(m, padded_at<kHalf>(row, c));
    m = asc::wave_max(m);
    __syncthreads();
    if ((t & 63) == 0) red[0][t >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    float s = 0.f;
    for (int64_t c = t; c < cols; c += 256) s += exp_nonpos(padded_at<kHalf>(row, c) - m);
    s = asc::wave_sum(s);
    if ((t & 63) == 0) red[1][t >> 6] = s;
    __syncthreads();
    s = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    s += static_cast<float>(pad) * exp_nonpos(0.0f - m);
    const float rs = 1.0f / s;
    for (int64_t c = t; c < cols; c += 256) {
      const float v = exp_nonpos(padded_at<kHalf>(row, c) - m) * rs;
      if constexpr (kHalf) static_cast<uint16_t*>(out)[r * stride + c] = to_half(v);
      else static_cast<float*>(out)[r * stride + c] = v;
    }
  }
}

}  // namespace softmax
}  // namespace asc

// Defines the softmax kernels, one per body, as `PREFIX##<body name>` with the
// given linkage specifier (the library's are internal, the code object's have C
// names for hipModuleGetFunction).  The names and their order are those of
// softmax.hip's kernel tables.
#define ASC_SOFTMAX_KERNEL(LINKAGE, NAME, THREADS, BODY) ASC_SOFTMAX_KERNEL_W(LINKAGE, NAME, THREADS, 1, BODY)
// WAVES: waves per SIMD that the registers must leave room for.
#define ASC_SOFTMAX_KERNEL_W(LINKAGE, NAME, THREADS, WAVES, BODY)                                                   \
  LINKAGE __global__ void __launch_bounds__(THREADS, WAVES)                                                               \
      NAME(const void* __restrict__ x, void* __restrict__ out, int64_t rows, int64_t stride, int32_t len,          \
           int32_t flag) {                                                                                         \
    BODY(x, out, rows, stride, len, flag);                                                                         \
  }

#define ASC_SOFTMAX_KERNELS(LINKAGE, PREFIX)                                                                       \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##wave_1x2, 256, (asc::softmax::wave_body<1, 2>))                              \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##wave_2x2, 256, (asc::softmax::wave_body<2, 2>))                              \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##block_2x128, 128, (asc::softmax::block_body<2, 128>))                        \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##block_2x256, 256, (asc::softmax::block_body<2, 256>))                        \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##block_2x512, 512, (asc::softmax::block_body<2, 512>))                        \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##block_8x256, 256, (asc::softmax::block_body<8, 256>))                        \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##long, 256, asc::softmax::long_body)                                          \
  ASC_SOFTMAX_KERNEL_W(LINKAGE, PREFIX##f16, 256, 4, asc::softmax::f16_body)                                            \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##padded_f32, 256, asc::softmax::padded_body<false>)                           \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##padded_f16, 256, asc::softmax::padded_body<true>)                            \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##short_f32, 256, asc::softmax::short_body)                                    \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##wide_f32, 1024, asc::softmax::wide_body)                                     \
  ASC_SOFTMAX_KERNEL(LINKAGE, PREFIX##wide_f16, 1024, asc::softmax::f16_wide_body)
