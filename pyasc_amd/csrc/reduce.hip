// Row reductions and RMS norm.
//
// asc_reduce_f32 covers the reference's reduction tests
// (python/test/asc2/operations/test_reduce_ops.py): asc2.reduce_{sum,max,min,prod}
// (python/asc/language/tile/reduction_ops.py:61-126) of a 2-D fp32 tile along
// dim 1 (one result per row), dim 0 (one per column) or over all elements
// (the scalar broadcast into an output by asc2.full).  fp32 accumulation; max
// and min return the larger / smaller non-NaN operand (IEEE maxNum / minNum).
//   dim 1: a wave per row, or a workgroup per row when there are few long rows; 16-byte
//          loads at element alignment, in-lane accumulation, DPP/permlane combine
//          (HBM-bound: 4 B per element).
//   dim 0: a workgroup per 64 columns walks the rows, 64 at a time, 16 bytes per lane; a
//          thread per four columns where rows are few or columns very many.
//   all:   one 1024-thread block.
// Few results leave most CUs idle: asc_reduce_f32_ws, with a workspace, splits the rows (dim
// 0) or the elements (all) over enough workgroups to fill the chip, and a second launch
// combines their partial results in a fixed order.
//
// asc_rms_norm covers asc2.rms_norm (python/asc/language/tile/unary_ops.py:225-237,
// AscendC RmsNorm): y = x * rsqrt(mean(x^2) + eps) * gamma along the last dim,
// fp32 or fp16 rows computed in fp32 (a block per row, the row held in
// registers up to 8192 fp32 / 16384 fp16 columns, two 16-byte vectors per lane
// from 1024 fp32 / 2048 fp16 columns up).
#include <math.h>

#include <type_traits>

#include "common.h"
#include "numeric.h"

namespace {

enum ReduceOp { kSum = 0, kMax = 1, kMin = 2, kProd = 3 };

template <int kOp>
__host__ __device__ constexpr float identity() {
  return kOp == kSum ? 0.0f : kOp == kMax ? -INFINITY : kOp == kMin ? INFINITY : 1.0f;
}

template <int kOp, class T>
__device__ __forceinline__ T combine(T a, T b) {
  if constexpr (kOp == kSum) return a + b;
  if constexpr (kOp == kMax) return fmaxf(a, b);
  if constexpr (kOp == kMin) return fminf(a, b);
  return a * b;
}

// Wave-wide combine; every lane ends with the same value (see asc::wave_sum).
template <int kOp>
__device__ __forceinline__ float wave_combine(float v) {
  v = combine<kOp>(v, asc::dpp_mov<asc::kDppQuadXor1>(v));
  v = combine<kOp>(v, asc::dpp_mov<asc::kDppQuadXor2>(v));
  v = combine<kOp>(v, asc::dpp_mov<asc::kDppRowHalfMirror>(v));
  v = combine<kOp>(v, asc::dpp_mov<asc::kDppRowMirror>(v));
  v = combine<kOp>(v, asc::lane_xor16(v));
  return combine<kOp>(v, asc::lane_xor32(v));
}

struct ReduceArgs {
  const float* x;
  float* out;
  int64_t rows, cols;
  int64_t out_count;  // "all": number of output elements receiving the result
  int64_t splits;     // dim 0, "all": workgroups that share one result's rows or elements
};

// First element of span i of n elements in `spans` parts, a multiple of 4.
__device__ __forceinline__ int64_t span_start(int64_t n, int64_t i, int64_t spans) {
  const int64_t vecs = n / 4;
  if (spans == 1) return i == 0 ? 0 : n;  // without the divisions, 0.4 us of a small launch
  return i == spans ? n : (vecs / spans * i + vecs % spans * i / spans) * 4;
}

// 16 bytes of fp32 at element alignment; kStream: read once, not kept in the caches.
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
template <bool kStream = true>
__device__ __forceinline__ f32x4_u load4(const float* p) {
  if constexpr (kStream) return __builtin_nontemporal_load(reinterpret_cast<const f32x4_u*>(p));
  return *reinterpret_cast<const f32x4_u*>(p);
}

// Elements [0, len) of x by the kThreads threads of a group (t: the thread's index in it):
// four independent vector loads per lane in flight, in-lane partials combined in a fixed order.
// What is left, at most four vectors per thread, is loaded at once too, each into a chain of its
// own, and the up to three elements behind the last vector join those of the first lanes.  Up to
// 64 elements take 16 lanes with up to four each: an element that only joins at the top of the
// tree would round once more at the full sum's size.
template <int kOp, int kThreads, class Int>
__device__ __forceinline__ float reduce_span(const float* x, Int len, int t) {
  constexpr int kUnroll = 4;
  float acc[4] = {identity<kOp>(), identity<kOp>(), identity<kOp>(), identity<kOp>()};
  const auto total = [&] { return combine<kOp>(combine<kOp>(acc[0], acc[1]), combine<kOp>(acc[2], acc[3])); };
  if (len <= 64) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (len > 16 * u && t < 16 && t + 16 * u < len) acc[u] = x[t + 16 * u];
    return total();
  }
  const auto add4 = [&](int u, f32x4_u v) {
    acc[u] = combine<kOp>(acc[u], combine<kOp>(combine<kOp>(v.x, v.y), combine<kOp>(v.z, v.w)));
  };
  const Int nvec = len / 4;
  Int q0 = 0;  // vectors taken by the whole group
  for (; q0 + kUnroll * kThreads <= nvec; q0 += kUnroll * kThreads) {
    f32x4_u v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] = load4(x + 4 * (q0 + t + u * kThreads));
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) add4(u, v[u]);
  }
  const int left = static_cast<int>(nvec - q0), rest = static_cast<int>(len - nvec * 4);
  constexpr float kId = identity<kOp>();
  const float tail = t < rest ? x[nvec * 4 + t] : kId;
  f32x4_u v[kUnroll];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    if (u > 0 && left <= u * kThreads) break;  // uniform
    v[u] = f32x4_u{kId, kId, kId, kId};
    if (t + u * kThreads < left) v[u] = load4(x + 4 * (q0 + t + u * kThreads));
  }
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    if (u > 0 && left <= u * kThreads) break;
    add4(u, v[u]);
  }
  acc[3] = combine<kOp>(acc[3], tail);
  return total();
}

// Combines one value per thread of a kThreads-thread workgroup; every thread gets the result.
// The waves' sums are added in pairs, the last four in fp64: a chain of sixteen fp32 additions was
// the largest part of a long row's rounding error (relative error against fp64, 300x65536: 6.0e-8
// with the chain, 4.4e-8 with one wave per row, 2.9e-8 with all of them in fp64).
template <int kOp, int kThreads>
__device__ __forceinline__ float block_combine(float v) {
  constexpr int kWaves = kThreads / 64;
  __shared__ float part[kWaves];
  v = wave_combine<kOp>(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  float p[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) p[w] = part[w];
#pragma unroll
  for (int n = kWaves / 2; n >= 4; n /= 2)
#pragma unroll
    for (int w = 0; w < n; ++w) p[w] = combine<kOp>(p[w], p[w + n]);
  using Part = std::conditional_t<kOp == kSum, double, float>;
  const Part lo = combine<kOp, Part>(p[0], p[1]), hi = combine<kOp, Part>(p[2], p[3]);
  return static_cast<float>(combine<kOp>(lo, hi));
}

// dim 1, a wave per row: rows 4*blockIdx.x + wave.
template <int kOp>
__global__ void __launch_bounds__(256) reduce_rows_kernel(ReduceArgs p) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= p.rows) return;
  const int len = static_cast<int>(p.cols);
  const float total = wave_combine<kOp>(reduce_span<kOp, 64>(p.x + r * p.cols, len, threadIdx.x & 63));
  if ((threadIdx.x & 63) == 0) p.out[r] = total;
}

// dim 1, a workgroup per row.
template <int kOp>
__global__ void __launch_bounds__(1024) reduce_long_rows_kernel(ReduceArgs p) {
  const int64_t r = blockIdx.x;
  const int len = static_cast<int>(p.cols);
  const float total = block_combine<kOp, 1024>(reduce_span<kOp, 1024>(p.x + r * p.cols, len, threadIdx.x));
  if (threadIdx.x == 0) p.out[r] = total;
}

// dim 0: workgroup (b, s) reduces rows [s*p.rows/splits, (s+1)*p.rows/splits) of columns 64b ..
// 64b+63 into out[s * cols + column].  Sixteen lanes cover 256 bytes of a row, a pass of the
// workgroup 64 rows, four passes' loads in flight.  Bound by HBM once every CU has a
// workgroup: 16384x4096 47-49 us (5.5-5.7 TB/s) with 256 workgroups of 64 columns, 57 with 32
// columns (128-byte pieces of rows), 69 with 128 workgroups; 65536x1024 47-51 us.  A thread per
// column took 6129 and 25088 us: one load in flight on 16 and 4 workgroups.
constexpr int kColsPerBlock = 64;
template <int kOp>
__global__ void __launch_bounds__(1024) reduce_cols_kernel(ReduceArgs p) {
  __shared__ float4 part[16][16];
  const int t = threadIdx.x, lane_c = t & 15;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kColsPerBlock + lane_c * 4;
  const int64_t r0 = p.rows * blockIdx.y / p.splits, r1 = p.rows * (blockIdx.y + 1) / p.splits;
  const int left = static_cast<int>(p.cols - c < 4 ? p.cols - c : 4);  // columns of this lane
  float acc[4] = {identity<kOp>(), identity<kOp>(), identity<kOp>(), identity<kOp>()};
  int64_t r = r0 + (t >> 4);
  if (left == 4) {
    const float* x = p.x + c;
    constexpr int kUnroll = 4;
    for (; r + (kUnroll - 1) * 64 < r1; r += kUnroll * 64) {
      f32x4_u v[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) v[u] = load4(x + (r + u * 64) * p.cols);
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = combine<kOp>(acc[i], v[u][i]);
    }
    for (; r < r1; r += 64) {
      const f32x4_u v = load4(x + r * p.cols);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = combine<kOp>(acc[i], v[i]);
    }
  } else if (left > 0) {
    for (; r < r1; r += 64)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i < left) acc[i] = combine<kOp>(acc[i], p.x[r * p.cols + c + i]);
  }
  // the wave's four rows, then the sixteen waves
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc[i] = combine<kOp>(acc[i], asc::lane_xor16(acc[i]));
    acc[i] = combine<kOp>(acc[i], asc::lane_xor32(acc[i]));
  }
  if ((t & 63) < 16) part[t >> 6][lane_c] = make_float4(acc[0], acc[1], acc[2], acc[3]);
  __syncthreads();
  if (t < kColsPerBlock) {
    const float* column = reinterpret_cast<const float*>(part) + t;
    float total = column[0];
#pragma unroll
    for (int w = 1; w < 16; ++w) total = combine<kOp>(total, column[w * kColsPerBlock]);
    const int64_t out_c = static_cast<int64_t>(blockIdx.x) * kColsPerBlock + t;
    if (out_c < p.cols) p.out[blockIdx.y * p.cols + out_c] = total;
  }
}

// dim 0 of few rows or very many columns: four columns per thread, eight rows' loads in flight,
// the last rows' at once too, one 16-byte store.  kStream only where x is larger than the L2s and
// made of aligned vectors: a smaller x may be in the L2 from its producer, and two threads share
// the lines of a misaligned row.  us, a thread per column before, here, x in the L2 / x from HBM:
// 31x65537 4.5, 4.6 / 14.1, 6.0; 20x262144 3.7, 2.8 / 10.7, 5.9; 31x1000003 23.2, 24.5 / 36, 29;
// 1x4194304 6.4, 4.9 / 11.3, 7.8; 24x4194304 (streamed) 107, 84 / 113, 84.
template <int kOp, bool kStream>
__global__ void __launch_bounds__(256) reduce_wide_cols_kernel(ReduceArgs p) {
  const int64_t c = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (c >= p.cols) return;
  float acc[4] = {identity<kOp>(), identity<kOp>(), identity<kOp>(), identity<kOp>()};
  const int left = static_cast<int>(p.cols - c < 4 ? p.cols - c : 4);
  const float* x = p.x + c;
  if (left < 4) {
    for (int64_t r = 0; r < p.rows; ++r)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i < left) acc[i] = combine<kOp>(acc[i], x[r * p.cols + i]);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < left) p.out[c + i] = acc[i];
    return;
  }
  const auto take = [&](f32x4_u v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = combine<kOp>(acc[i], v[i]);
  };
  constexpr int kUnroll = 8;
  int64_t r = 0;
  f32x4_u v[kUnroll];
  for (; r + kUnroll <= p.rows; r += kUnroll) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] = load4<kStream>(x + (r + u) * p.cols);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) take(v[u]);
  }
  const int rest = static_cast<int>(p.rows - r);
#pragma unroll
  for (int u = 0; u < kUnroll - 1; ++u)
    if (u < rest) v[u] = load4<kStream>(x + (r + u) * p.cols);
#pragma unroll
  for (int u = 0; u < kUnroll - 1; ++u)
    if (u < rest) take(v[u]);
  *reinterpret_cast<f32x4_u*>(p.out + c) = f32x4_u{acc[0], acc[1], acc[2], acc[3]};
}

// all elements: workgroup s reduces elements [s*n/grid, (s+1)*n/grid); the result is written to
// out[0 .. out_count), or with several workgroups to out[s].
template <int kOp>
__global__ void __launch_bounds__(1024) reduce_all_kernel(ReduceArgs p) {
  const int64_t n = p.rows * p.cols;
  const int64_t e0 = span_start(n, blockIdx.x, p.splits), e1 = span_start(n, blockIdx.x + 1, p.splits);
  const float total = block_combine<kOp, 1024>(reduce_span<kOp, 1024>(p.x + e0, e1 - e0, threadIdx.x));
  if (p.splits > 1) {
    if (threadIdx.x == 0) p.out[blockIdx.x] = total;
    return;
  }
  for (int64_t i = threadIdx.x; i < p.out_count; i += 1024) p.out[i] = total;
}

// dim 0 by a thread per four columns: with fewer than 32 rows most of a 64-row pass would be
// idle, and from 2^18 columns up those threads fill the chip.
bool wide_cols(int64_t rows, int64_t cols) { return rows < 32 || cols >= (int64_t{1} << 18); }

// Workgroups that a reduction's rows (dim 0) or elements (all) are split over when it has a
// workspace; 1: no second launch.  A second launch costs about 3 us: it pays from about 1 MiB
// of input.  256 workgroups, one per CU, are as fast as more of them (16384x4096, column sums
// and all elements: 47.1 and 44.9 us with 256, 48.7 and 47.9 with 512).
constexpr int64_t kSplitMinElems = int64_t{1} << 18;
constexpr int64_t kSplitGroups = 256;
int64_t reduce_splits(int64_t rows, int64_t cols, int dim) {
  const int64_t n = rows * cols;
  if (n < kSplitMinElems || dim == 1) return 1;
  if (dim == -1) return n / 16384 < kSplitGroups ? n / 16384 : kSplitGroups;
  if (wide_cols(rows, cols)) return 1;
  const int64_t col_groups = asc::ceil_div(cols, kColsPerBlock);
  const int64_t by_groups = kSplitGroups / col_groups, by_rows = rows / 512;
  const int64_t splits = by_groups < by_rows ? by_groups : by_rows;
  return splits < 1 ? 1 : splits;
}

template <int kOp>
void launch_cols(const ReduceArgs& p, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>(asc::ceil_div(p.cols, kColsPerBlock)), static_cast<uint32_t>(p.splits));
  hipLaunchKernelGGL(reduce_cols_kernel<kOp>, grid, dim3(1024), 0, s, p);
}

template <int kOp>
void launch_wide_cols(const ReduceArgs& p, hipStream_t s) {
  // a wave per workgroup spreads fewer than 2^18 columns over the CUs (31x65537: 4.6 us, 5.3 with
  // four); past that four are the better (31x1000003: 27.7 us with one, 24.5)
  const int threads = p.cols < (int64_t{1} << 18) ? 64 : 256;
  const bool stream = asc::aligned16(p.x) && p.cols % 4 == 0 && p.rows * p.cols > (int64_t{8} << 20);
  const auto kernel = stream ? reduce_wide_cols_kernel<kOp, true> : reduce_wide_cols_kernel<kOp, false>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(asc::ceil_div(p.cols, 4 * threads))), dim3(threads), 0, s, p);
}

// ws: room for the partial results of p.splits groups (null: p.splits is 1)
template <int kOp>
int32_t launch_reduce(const ReduceArgs& p, int dim, float* ws, hipStream_t s) {
  if (dim == 1) {
    // A wave per row keeps HBM busy from about 1024 rows up (16384x4096: 6.0 TB/s).  Fewer rows of
    // 2048 columns or more take a workgroup each while the rows are long for their number: us with a
    // wave, a workgroup, x from HBM: 512x2048 3.1, 2.7; 768x4096 4.6, 4.5; 1023x2048 3.5, 4.1;
    // 1023x8192 8.2, 7.7.  One dispatch covers fewer than 2^32 threads.
    const bool wave_rows = p.rows >= 1024 || p.cols < 2048 || p.cols < 4 * p.rows;
    const int64_t blocks = wave_rows ? asc::ceil_div(p.rows, 4) : p.rows;
    ASC_REQUIRE(blocks * 256 < (int64_t{1} << 32), ASC_ERR_UNSUPPORTED, "asc_reduce_f32: %lld rows exceed one launch",
                static_cast<long long>(p.rows));
    if (wave_rows) {
      hipLaunchKernelGGL(reduce_rows_kernel<kOp>, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, p);
    } else {
      hipLaunchKernelGGL(reduce_long_rows_kernel<kOp>, dim3(static_cast<uint32_t>(blocks)), dim3(1024), 0, s, p);
    }
  } else if (dim == 0) {
    if (wide_cols(p.rows, p.cols)) {
      launch_wide_cols<kOp>(p, s);
    } else if (p.splits == 1) {
      launch_cols<kOp>(p, s);
    } else {
      launch_cols<kOp>(ReduceArgs{p.x, ws, p.rows, p.cols, 0, p.splits}, s);
      launch_cols<kOp>(ReduceArgs{ws, p.out, p.splits, p.cols, 0, 1}, s);
    }
  } else if (p.splits == 1) {
    hipLaunchKernelGGL(reduce_all_kernel<kOp>, dim3(1), dim3(1024), 0, s, p);
  } else {
    hipLaunchKernelGGL(reduce_all_kernel<kOp>, dim3(static_cast<uint32_t>(p.splits)), dim3(1024), 0, s,
                       ReduceArgs{p.x, ws, p.rows, p.cols, 0, p.splits});
    hipLaunchKernelGGL(reduce_all_kernel<kOp>, dim3(1), dim3(1024), 0, s,
                       ReduceArgs{ws, p.out, 1, p.splits, p.out_count, 1});
  }
  return asc::check_launch("asc_reduce_f32");
}

// ---- RMS norm

struct F32E {
  using T = float;
  static constexpr int kPerVec = 4;
};
struct F16E {
  using T = uint16_t;
  static constexpr int kPerVec = 8;
};

struct RmsArgs {
  const void* x;
  const float* gamma;
  void* out;
  int64_t rows, stride;  // stride = num_cols (elements between row starts)
  int32_t len;           // columns normalised per row
  float eps;
  bool vec_ok;
};

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// 16-byte vector q of a row as fp32 values (0 past len).
template <class E>
__device__ __forceinline__ void load_elems(const typename E::T* row, int q, int len, bool full, float (&v)[E::kPerVec]) {
  constexpr int kP = E::kPerVec;
  const int e = q * kP;
  if (full) {
    const u32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row) + q);
    typename E::T t[kP];
    __builtin_memcpy(t, &raw, 16);
#pragma unroll
    for (int i = 0; i < kP; ++i) {
      if constexpr (sizeof(typename E::T) == 4) v[i] = t[i];
      else v[i] = asc::f16_to_f32(t[i]);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < kP; ++i) {
    float f = 0.0f;
    if (e + i < len) {
      if constexpr (sizeof(typename E::T) == 4) f = row[e + i];
      else f = asc::f16_to_f32(row[e + i]);
    }
    v[i] = f;
  }
}

template <class E>
__device__ __forceinline__ void store_elems(typename E::T* row, int q, int len, bool full,
                                            const float (&v)[E::kPerVec]) {
  constexpr int kP = E::kPerVec;
  typename E::T t[kP];
#pragma unroll
  for (int i = 0; i < kP; ++i) {
    if constexpr (sizeof(typename E::T) == 4) t[i] = v[i];
    else t[i] = asc::f32_to_f16_rne(v[i]);
  }
  if (full) {
    u32x4 raw;
    __builtin_memcpy(&raw, t, 16);
    __builtin_nontemporal_store(raw, reinterpret_cast<u32x4*>(row) + q);
    return;
  }
  const int e = q * kP;
#pragma unroll
  for (int i = 0; i < kP; ++i)
    if (e + i < len) row[e + i] = t[i];
}

// y = (x * inv_rms) * gamma, inv_rms = 1 / sqrt(sum(x^2) / len + eps)
// (correctly rounded division and square root).  kThreads threads per row,
// VPT 16-byte vectors per thread; gamma is read as 16-byte vectors too.
template <class E, int VPT, int kThreads>
__global__ void __launch_bounds__(kThreads) rms_norm_kernel(RmsArgs p) {
  using T = typename E::T;
  constexpr int kP = E::kPerVec;
  constexpr int kWaves = kThreads / 64;
  __shared__ float red[kWaves];
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x;
  const T* xr = static_cast<const T*>(p.x) + r * p.stride;
  T* orow = static_cast<T*>(p.out) + r * p.stride;
  float v[VPT][kP];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    // uniform test: vector j is inside the row for every thread
    const bool full = p.vec_ok && kThreads * (j + 1) * kP <= p.len;
    load_elems<E>(xr, t + kThreads * j, p.len, full, v[j]);
  }
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
#pragma unroll
    for (int i = 0; i < kP; ++i) ss += v[j][i] * v[j][i];
  ss = asc::wave_sum(ss);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  float total = red[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) total += red[w];
  const float inv = 1.0f / sqrtf(total / static_cast<float>(p.len) + p.eps);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int q = t + kThreads * j;
    const bool full = p.vec_ok && kThreads * (j + 1) * kP <= p.len;
    float gm[kP];
    if (full) {
#pragma unroll
      for (int h = 0; h < kP / 4; ++h) {
        const u32x4 g4 = *reinterpret_cast<const u32x4*>(p.gamma + q * kP + 4 * h);
        __builtin_memcpy(gm + 4 * h, &g4, 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kP; ++i) gm[i] = q * kP + i < p.len ? p.gamma[q * kP + i] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kP; ++i) v[j][i] = (v[j][i] * inv) * gm[i];
    store_elems<E>(orow, q, p.len, full, v[j]);
  }
}

// Rows longer than the register-resident variant: two passes over the row.
template <class E>
__global__ void __launch_bounds__(256) rms_norm_long_kernel(RmsArgs p) {
  using T = typename E::T;
  __shared__ float red[4];
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x;
  const T* xr = static_cast<const T*>(p.x) + r * p.stride;
  T* orow = static_cast<T*>(p.out) + r * p.stride;
  auto at = [&](int c) -> float {
    if constexpr (sizeof(T) == 4) return xr[c];
    else return asc::f16_to_f32(xr[c]);
  };
  float ss = 0.0f;
  for (int c = t; c < p.len; c += 256) {
    const float x = at(c);
    ss += x * x;
  }
  ss = asc::wave_sum(ss);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  const float total = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = 1.0f / sqrtf(total / static_cast<float>(p.len) + p.eps);
  for (int c = t; c < p.len; c += 256) {
    const float y = (at(c) * inv) * p.gamma[c];
    if constexpr (sizeof(T) == 4) orow[c] = y;
    else orow[c] = asc::f32_to_f16_rne(y);
  }
}

template <class E>
int32_t launch_rms(const RmsArgs& p, hipStream_t s) {
  constexpr int kP = E::kPerVec;
  // One workgroup per row, two 16-byte vectors per lane above 256 vectors per row:
  // more, shorter waves per row finish each row's loads, reduction and stores sooner
  // (4096 fp32 columns, 64 MiB in and out, same box: 5480-5530 GB/s with 128 threads
  // x 8 vectors, 5730-5740 with 512 x 2, 5040 with 1024 x 1; 2048 columns: 5500-5550
  // with 128 x 4, 5650-5680 with 256 x 2; 8192: 5370 with 256 x 8, 5510 with 512 x 4,
  // 5560-5570 with 1024 x 2).  Two passes over longer rows.
  const int64_t vecs = (static_cast<int64_t>(p.len) + kP - 1) / kP;
  const int64_t threads = vecs <= 256 ? 128 : vecs <= 512 ? 256 : vecs <= 1024 ? 512 : vecs <= 2048 ? 1024 : 256;
  // one dispatch covers fewer than 2^32 threads
  ASC_REQUIRE(p.rows * threads < (int64_t{1} << 32), ASC_ERR_UNSUPPORTED, "asc_rms_norm: %lld rows exceed one launch",
              static_cast<long long>(p.rows));
  const dim3 grid(static_cast<uint32_t>(p.rows));
  if (vecs <= 128) {
    hipLaunchKernelGGL((rms_norm_kernel<E, 1, 128>), grid, dim3(128), 0, s, p);
  } else if (vecs <= 256) {
    hipLaunchKernelGGL((rms_norm_kernel<E, 2, 128>), grid, dim3(128), 0, s, p);
  } else if (vecs <= 512) {
    hipLaunchKernelGGL((rms_norm_kernel<E, 2, 256>), grid, dim3(256), 0, s, p);
  } else if (vecs <= 1024) {
    hipLaunchKernelGGL((rms_norm_kernel<E, 2, 512>), grid, dim3(512), 0, s, p);
  } else if (vecs <= 2048) {
    hipLaunchKernelGGL((rms_norm_kernel<E, 2, 1024>), grid, dim3(1024), 0, s, p);
  } else {
    hipLaunchKernelGGL(rms_norm_long_kernel<E>, grid, dim3(256), 0, s, p);
  }
  return asc::check_launch("asc_rms_norm");
}

}  // namespace

extern "C" int32_t asc_reduce_f32_ws(int32_t op, const float* x, float* out, int64_t rows, int64_t cols, int32_t dim,
                                     int64_t out_count, void* workspace, int64_t workspace_bytes,
                                     asc_stream_t stream) {
  ASC_REQUIRE(op >= kSum && op <= kProd, ASC_ERR_INVALID_ARG, "asc_reduce_f32: op must be 0..3, got %d", op);
  ASC_REQUIRE(dim == 0 || dim == 1 || dim == -1, ASC_ERR_INVALID_ARG,
              "asc_reduce_f32: dim must be 0, 1 or -1 (all), got %d", dim);
  ASC_REQUIRE(rows >= 0 && cols >= 0 && out_count >= 0, ASC_ERR_INVALID_ARG, "asc_reduce_f32: negative size");
  ASC_REQUIRE(cols < (int64_t{1} << 31), ASC_ERR_UNSUPPORTED, "asc_reduce_f32: cols too large");
  const int64_t results = dim == 1 ? rows : dim == 0 ? cols : out_count;
  if (results == 0) return ASC_OK;
  ASC_REQUIRE(rows > 0 && cols > 0, ASC_ERR_INVALID_ARG, "asc_reduce_f32: empty input");
  ASC_REQUIRE(x && out, ASC_ERR_INVALID_ARG, "asc_reduce_f32: null buffer");
  ReduceArgs p{x, out, rows, cols, out_count, 1};
  if (workspace != nullptr) {
    p.splits = reduce_splits(rows, cols, dim);
    const int64_t need = asc_reduce_f32_workspace(rows, cols, dim);
    ASC_REQUIRE(workspace_bytes >= need, ASC_ERR_INVALID_ARG,
                "asc_reduce_f32_ws: the partial results need %lld bytes, the workspace holds %lld", (long long)need,
                (long long)workspace_bytes);
    ASC_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 3) == 0, ASC_ERR_ALIGNMENT,
                "asc_reduce_f32_ws: the workspace must be 4-byte aligned");
  }
  float* ws = static_cast<float*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (op) {
    case kSum: return launch_reduce<kSum>(p, dim, ws, s);
    case kMax: return launch_reduce<kMax>(p, dim, ws, s);
    case kMin: return launch_reduce<kMin>(p, dim, ws, s);
    default: return launch_reduce<kProd>(p, dim, ws, s);
  }
}

extern "C" int32_t asc_reduce_f32_workspace(int64_t rows, int64_t cols, int32_t dim) {
  if (rows <= 0 || cols <= 0) return 0;
  const int64_t splits = reduce_splits(rows, cols, dim);
  // dim 0: splits * ceil(cols / 64) <= 256, so this never exceeds 64 KiB
  return splits == 1 ? 0 : static_cast<int32_t>(splits * (dim == 0 ? cols : 1) * static_cast<int64_t>(sizeof(float)));
}

extern "C" int32_t asc_reduce_f32(int32_t op, const float* x, float* out, int64_t rows, int64_t cols, int32_t dim,
                                  int64_t out_count, asc_stream_t stream) {
  return asc_reduce_f32_ws(op, x, out, rows, cols, dim, out_count, nullptr, 0, stream);
}

extern "C" int32_t asc_rms_norm(int32_t dtype, const void* x, const float* gamma, void* out, int64_t num_rows,
                                int64_t num_cols, int32_t tile_size, float epsilon, asc_stream_t stream) {
  ASC_REQUIRE(num_rows >= 0 && num_cols >= 0, ASC_ERR_INVALID_ARG, "asc_rms_norm: negative shape");
  ASC_REQUIRE(tile_size > 0 && tile_size <= num_cols, ASC_ERR_INVALID_ARG,
              "asc_rms_norm: need 0 < tile_size <= num_cols (got %d, %lld)", tile_size, (long long)num_cols);
  ASC_REQUIRE(dtype == ASC_DT_FLOAT32 || dtype == ASC_DT_FLOAT16, ASC_ERR_UNSUPPORTED,
              "asc_rms_norm: dtype %d not supported (float32, float16)", dtype);
  if (num_rows == 0) return ASC_OK;
  ASC_REQUIRE(x && gamma && out, ASC_ERR_INVALID_ARG, "asc_rms_norm: null buffer");
  const int64_t es = dtype == ASC_DT_FLOAT32 ? 4 : 2;
  RmsArgs p{x, gamma, out, num_rows, num_cols, tile_size, epsilon,
            asc::aligned16(x) && asc::aligned16(out) && asc::aligned16(gamma) && (num_cols * es) % 16 == 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == ASC_DT_FLOAT32 ? launch_rms<F32E>(p, s) : launch_rms<F16E>(p, s);
}
