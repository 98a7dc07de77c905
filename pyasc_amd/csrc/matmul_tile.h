// The tile kernels (gemm_tile.h) of the matmuls: their variants, the element types they
// are built for and the host-side choice among them, shared by matmul.hip (fp16, bf16,
// fp32 inputs) and matmul_i8.hip (int8).
#pragma once

#include "gemm_tile.h"
#include "matmul_i8_kernels.h"
#include "matmul_kernels.h"

namespace asc {
namespace tile {

using asc::gemm::TileArgs;
using asc::gemm::u32x4;

// fp32 accumulators: bias, activation and cast as asc::mm::Epilogue.
struct FloatOut {
  using Val = float;
  static constexpr bool kInt = false;
  __device__ __forceinline__ static float vec_at(const TileArgs& p, int n) {
    return p.vec != nullptr ? p.vec[n] : 0.0f;
  }
  template <int kOut>
  __device__ __forceinline__ static uint32_t out_bits(float v, float vec_n, const TileArgs& p) {
    // The activation is uniform, but as a lane value it becomes two selects per element: a
    // branch per element and activation made the epilogue longer than the main loop.
    int act = p.act;
    asm("" : "+v"(act));
    if (p.vec != nullptr) v += vec_n;
    const float relu = fmaxf(v, 0.0f), leaky = v >= 0.0f ? v : v * p.alpha;
    v = act == 1 ? relu : act == 2 ? leaky : v;
    if constexpr (kOut == asc::gemm::kTileOutF32) return __float_as_uint(v);
    else if constexpr (kOut == asc::gemm::kTileOutF16) return asc::f32_to_f16_rne(v);
    else return asc::f32_to_bf16_rne(v);
  }
};

template <bool kBf16>
struct Tr16 : FloatOut {
  using Elem = uint16_t;
  using Acc = asc::mm::f32x16;
  __device__ __forceinline__ static Acc mfma(u32x4 a, u32x4 b, Acc c) { return asc::mm::Tr16<kBf16>::mfma(a, b, c); }
};

// fp32: a chunk of 4 values per lane half takes four v_mfma_f32_32x32x2_f32 (A and B pair the
// same k), each into an accumulator of its own: four chains a quarter as long, summed at the
// end, keep the rounding error below that of a kernel that splits K over four waves
// (1024^3: 2.1e-7 relative to fp64 in the 2-norm, against 4.1e-7 with one chain; 21.5 us against
// 20.4).
struct TrF32 : FloatOut {
  using Elem = float;
  struct Acc {
    asc::mm::f32x16 part[4];
    __device__ __forceinline__ float operator[](int r) const {
      return (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
    }
  };
  __device__ __forceinline__ static Acc mfma(u32x4 a, u32x4 b, const Acc& c) {
    Acc d;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d.part[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e]), __uint_as_float(b[e]), c.part[e], 0, 0, 0);
    }
    return d;
  }
};

// int32 accumulators as they are, or the fp16 dequant: fp16_rne(fp32_rne(acc) * scale[n]).
struct TrI8 {
  using Elem = int8_t;
  using Acc = asc::i8::i32x16;
  using Val = int32_t;
  static constexpr bool kInt = true;
  __device__ __forceinline__ static Acc mfma(u32x4 a, u32x4 b, Acc c) { return asc::i8::TrI8::mfma(a, b, c); }
  __device__ __forceinline__ static float vec_at(const TileArgs& p, int n) {
    if (p.vec == nullptr) return 0.0f;
    const float s = p.vec[n];
    return p.trunc19 ? __uint_as_float(__float_as_uint(s) & 0xFFFFE000u) : s;
  }
  template <int kOut>
  __device__ __forceinline__ static uint32_t out_bits(int32_t x, float scale_n, const TileArgs&) {
    if constexpr (kOut == asc::gemm::kTileOutI32) return static_cast<uint32_t>(x);
    else return asc::f32_to_f16_rne(asc::materialize(static_cast<float>(x) * scale_n));
  }
};

// One kernel variant: its tile and workgroup, and its cost model.  A launch of T tiles over
// k-tiles of 64 bytes takes about ceil(T / 256) * (ktiles * per_ktile_us + fixed_us): 256 CUs
// hold one tile each (a CU that holds two takes about twice as long), and a round pays for
// filling its pipeline and storing its tile once.  per_ktile_us and fixed_us are fitted to
// measured launches (3 rotating operand sets, one MI355X); the choice only has to rank
// variants, and does so within about 10% on the shapes it was fitted to.
struct Variant {
  const char* name;  // in the kernels' names
  int bm, bn, threads;
  float per_ktile_us, fixed_us;
};

// fp16 / bf16 / int8 (an MFMA takes the same cycles per byte of K), 16-byte aligned
// operands.  Measured in us, bf16 unless noted:
//   1999x4096x4096: 128x256 65, 128x128 76, 256x256 87, 192x128 91
//   3000x3000x3000: 256x256 74, 192x128 80, 128x256 87, 128x128 91
//   333x11008x4096: 192x128 51, 128x256 57, 128x128 67, 256x256 84
//   600x4096x4096: 128x128 33, 192x128 44, 64x64 45, 128x256 48
//   1000x1000x1000: 64x64k2 8.7, 64x64 9.2, 32x64 12.4, 128x128 13.8
//   16x11008x4096: 32x64 17.5, 64x64k2 18.0, 32x32 25.4, 128x128 32.7
//   16x4096x11008: 32x32 33, 32x64 36, 64x64k2 39;  512x512x256: 32x32 3.7, 64x64 4.3
enum DmaVariant { kD256x256, kD128x256, kD192x128, kD128x128, kD64x64, kD64x64k2, kD32x64, kD32x32, kNumDma };
constexpr Variant kDma[kNumDma] = {{"256x256", 256, 256, 512, 0.85f, 6.0f}, {"128x256", 128, 256, 512, 0.51f, 5.0f},
                                   {"192x128", 192, 128, 512, 0.38f, 4.5f}, {"128x128", 128, 128, 512, 0.28f, 4.0f},
                                   {"64x64", 64, 64, 256, 0.10f, 2.2f},     {"64x64k2", 64, 64, 512, 0.10f, 2.0f},
                                   {"32x64", 32, 64, 512, 0.085f, 2.0f},    {"32x32", 32, 32, 256, 0.07f, 1.8f}};
// Any alignment (loads through registers).  1999x4097x4095: 256x256 126, 128x128 152, 64x64
// 211; 333x11007x4095: 128x128 86, 256x256 127, 64x64 127; 1000x1000x1001: 64x64 11,
// 128x128 19, 32x32 18; 17x1001x5003: 32x32 19, 64x64 30.
enum AnyVariant { kA256x256, kA128x128, kA64x64, kA32x32, kNumAny };
constexpr Variant kAny[kNumAny] = {{"any_256x256", 256, 256, 512, 0.95f, 6.0f},
                                   {"any_128x128", 128, 128, 512, 0.40f, 4.0f},
                                   {"any_64x64", 64, 64, 512, 0.23f, 2.2f},
                                   {"any_32x32", 32, 32, 256, 0.10f, 2.0f}};
// fp32: v_mfma_f32_32x32x2 takes 8 times the cycles per byte of K, so these are bound by the
// MFMAs and the tile hardly matters once the CUs are full.  2000^3: 128x128 133, 64x64 145,
// 32x32 154; 1024^3: 64x64 24, 32x32 24, 128x128 66; 256^3: 32x32 4.5, 64x64 7.9; any
// alignment 2001x2003x1999: 128x128 137, 64x64 144; 1001x999x1003: 64x64 25, 32x32 34.
enum F32Variant { kF128x128, kF64x64, kF32x32, kFA128x128, kFA64x64, kFA32x32, kNumF32 };
constexpr Variant kF32[kNumF32] = {{"128x128", 128, 128, 512, 0.97f, 4.0f},    {"64x64", 64, 64, 512, 0.30f, 2.2f},
                                   {"32x32", 32, 32, 256, 0.09f, 1.8f},        {"any_128x128", 128, 128, 512, 1.06f, 4.0f},
                                   {"any_64x64", 64, 64, 512, 0.35f, 2.2f},    {"any_32x32", 32, 32, 256, 0.13f, 2.0f}};

constexpr int kCus = 256;

// A launch of the 16x16-block kernel of matmul_kernels.h, in the units of the variants' models: a
// short start, then a chain of loads along K (with few rows most of A's are masked) or, with many
// blocks, the rate at which they get through K.  Against it the tiles' models, which rank tiles on
// products of some length, leave out part of their start.  The lines end where the tiles' time per
// k-tile is the smaller one throughout.  Measured us, blocks and tiles: 64x64x16 2.7, 3.4; 256x256x64
// 3.0, 3.5; 512x512x32 3.5, 3.7; 16x4096x128 3.7, 3.8; 1x64x256 3.3, 4.0; 256x256x256 4.9, 4.3;
// unaligned 260x260x57 2.9, 4.9; 300x301x100 3.6, 5.1; 113x1390x137 5.0, 6.0; 512x257x192 6.7, 5.7.
inline double f32_blocks_us(bool aligned, int64_t M, int64_t N, int64_t K) {
  const double blocks = static_cast<double>((M + 15) / 16) * static_cast<double>((N + 15) / 16);
  const double chain = M <= 8 ? 0.0052 : 0.011, rate = (aligned ? 3.4e-5 : 4.2e-5) * blocks;
  const double along_k = static_cast<double>(K) * (chain > rate ? chain : rate), starts = 0.0008 * blocks;
  return 0.8 + (along_k > starts ? along_k : starts);
}
inline bool f32_prefers_blocks(int index, double us, int64_t M, int64_t N, int64_t K) {
  constexpr double kStart[kNumF32] = {0.0, 0.4, 0.0, 0.0, 1.2, 1.8}, kLeast[kNumF32] = {0.0, 3.5, 2.3, 0.0, 0.0, 0.0};
  const bool aligned = index < kFA128x128;
  if (K > (M <= 8 ? 512 : aligned ? 160 : 320)) return false;
  const Variant& v = kF32[index];
  const int64_t tiles = ((M + v.bm - 1) / v.bm) * ((N + v.bn - 1) / v.bn);
  const double rounds = static_cast<double>((tiles + kCus - 1) / kCus);
  us += rounds * kStart[index];
  if (us < rounds * kLeast[index]) us = rounds * kLeast[index];
  return f32_blocks_us(aligned, M, N, K) <= us;
}

// One tile launch: the variant's index in its type's kernel table, name, arguments, grid.
struct TileLaunch {
  int index = -1;  // -1: no variant takes the call
  const char* name = nullptr;
  TileArgs p{};
  int64_t blocks = 0;
  int threads = 0;
  double us = 0.0;  // modelled time
};

// Picks among variants [first, last) of `table` the one with the least modelled time whose
// grid fits one launch and that `takes` accepts, and fills in tiles, grid and name.  K > 0.
template <class Takes>
inline void choose(const Variant* table, int first, int last, int64_t M, int64_t N, int64_t k_bytes, TileLaunch& L,
                   Takes takes) {
  const double ktiles = static_cast<double>(k_bytes) / 64.0;
  for (int i = first; i < last; ++i) {
    const Variant& v = table[i];
    const int64_t tm = (M + v.bm - 1) / v.bm, tn = (N + v.bn - 1) / v.bn, tiles = tm * tn;
    if (tiles * v.threads >= (int64_t{1} << 32) || tiles >= (int64_t{1} << 31) || !takes(i)) continue;
    const double us = static_cast<double>((tiles + kCus - 1) / kCus) * (ktiles * v.per_ktile_us + v.fixed_us);
    if (L.index >= 0 && us >= L.us) continue;
    L.us = us;
    L.index = i;
    L.name = v.name;
    L.blocks = tiles;
    L.threads = v.threads;
    L.p.tiles_m = static_cast<int>(tm);
    L.p.tiles_n = static_cast<int>(tn);
  }
}

// Whether C lies in place of an operand: rows of `c_bytes` and `bytes`, both `pitch` bytes apart,
// that start within one row of each other and share memory.
inline bool in_place(const void* x, int64_t pitch, int64_t bytes, const void* c, int64_t c_pitch, int64_t c_bytes) {
  if (pitch != c_pitch) return false;
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), c0 = reinterpret_cast<uintptr_t>(c);
  const int64_t shift = c0 >= x0 ? static_cast<int64_t>(c0 - x0) : -static_cast<int64_t>(x0 - c0);
  if (shift <= -pitch || shift >= pitch) return false;
  // C's row meets its own row of x, the next or the one before
  return (shift < bytes && shift + c_bytes > 0) || shift + c_bytes > pitch || shift + pitch < bytes;
}

// Whether the direct-to-LDS variants can address the operands: 16-byte chunks throughout, and
// offsets from a tile's first row or k-tile below the out-of-bounds mark of their 31 bits.
inline bool dma_takes(const void* a, const void* b, int64_t N, int64_t K, int64_t lda, int64_t ldb, int es) {
  constexpr int64_t kLimit = (int64_t{1} << 31) - (1 << 20);
  const uintptr_t at = reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b);
  return (at & 15) == 0 && ((lda | ldb | N | K) * es) % 16 == 0 && 256 * lda * es + K * es < kLimit &&
         128 * ldb * es < kLimit;
}

// Picks the variant for an fp16 / bf16 / int8 product (element size `es`); 64x64k2 splits K over
// two groups, which only helps while a CU holds one tile.  aligned256: the tile-aligned loop of
// gemm_direct.h takes the product (variant 256x256 stands for it).  From 129 of its tiles up, the
// larger tiles are better than the model says where a round leaves CUs idle, as the others share more
// of the L2 and of the power.  Up to 256 of its tiles that loop takes the product, above 192x128
// has to be 15% better by the model (us, the better of the loop and 128x256, and 192x128: bf16
// 3072x3072x4096 81, 93; 3072x4096x11008 232, 262; 6144x4096x11008 469, 518; 6144x6144x11008 783, 842;
// int8 3072x3072x11008 110, 127; but 4608x4096x4096 180, 157).
inline void choose_mfma(int es, bool dma, bool aligned256, int64_t M, int64_t N, int64_t K, TileLaunch& L) {
  if (dma) {
    const int64_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64), tiles256 = ((M + 255) / 256) * ((N + 255) / 256);
    const bool many = aligned256 && tiles256 > kCus / 2, one_round = many && tiles256 <= kCus;
    choose(kDma, 0, one_round ? kD256x256 + 1 : kNumDma, M, N, K * es, L, [&](int i) {
      return i == kD64x64 ? tiles64 > kCus : i == kD64x64k2 ? tiles64 <= kCus : !(many && i == kD192x128);
    });
    if (many && !one_round) {
      TileLaunch other;
      choose(kDma, kD192x128, kD192x128 + 1, M, N, K * es, other, [](int) { return true; });
      if (other.index >= 0 && L.index >= 0 && other.us < 0.85 * L.us) L = other;
    }
    return;
  }
  choose(kAny, 0, kNumAny, M, N, K * es, L, [](int) { return true; });
  if (L.index >= 0) L.index += kNumDma;
}

inline void choose_f32(bool dma, int64_t M, int64_t N, int64_t K, TileLaunch& L) {
  choose(kF32, dma ? 0 : kFA128x128, dma ? kFA128x128 : kNumF32, M, N, K * 4, L, [](int) { return true; });
}

}  // namespace tile
}  // namespace asc

// Defines (or, with ASC_TILE_DECLARE, declares) the tile kernels of one element type, each
// taking one TileArgs by value.  The template arguments are those of TileGemm:
// kI, kJ, kWM, kWN, kKW, kStages, kKB, kDma, kLean.
#define ASC_TILE_DEFINE(LINKAGE, NAME, TR, ...)                                                            \
  LINKAGE __global__ void __launch_bounds__((asc::gemm::TileGemm<TR, __VA_ARGS__>::kThreads))              \
      NAME(asc::gemm::TileArgs p) {                                                                        \
    asc::gemm::tile_body<asc::gemm::TileGemm<TR, __VA_ARGS__>, TR>(p);                                     \
  }
#define ASC_TILE_DECLARE(LINKAGE, NAME, TR, ...) LINKAGE __global__ void NAME(asc::gemm::TileArgs p);

#define ASC_TILE_KERNELS_MFMA(WHAT, LINKAGE, PREFIX, TR)                             \
  WHAT(LINKAGE, PREFIX##256x256, TR, 4, 2, 2, 4, 1, 5, 64, true, false)              \
  WHAT(LINKAGE, PREFIX##128x256, TR, 2, 2, 2, 4, 1, 3, 128, true, true)              \
  WHAT(LINKAGE, PREFIX##192x128, TR, 3, 1, 2, 4, 1, 3, 128, true, true)              \
  WHAT(LINKAGE, PREFIX##128x128, TR, 2, 1, 2, 4, 1, 4, 128, true, true)              \
  WHAT(LINKAGE, PREFIX##64x64, TR, 1, 1, 2, 2, 1, 4, 128, true, true)                \
  WHAT(LINKAGE, PREFIX##64x64k2, TR, 1, 1, 2, 2, 2, 4, 128, true, true)              \
  WHAT(LINKAGE, PREFIX##32x64, TR, 1, 1, 1, 2, 4, 4, 64, true, true)                 \
  WHAT(LINKAGE, PREFIX##32x32, TR, 1, 1, 1, 1, 4, 5, 64, true, true)                 \
  WHAT(LINKAGE, PREFIX##any_256x256, TR, 4, 2, 2, 4, 1, 2, 64, false, false)         \
  WHAT(LINKAGE, PREFIX##any_128x128, TR, 2, 1, 2, 4, 1, 4, 64, false, false)         \
  WHAT(LINKAGE, PREFIX##any_64x64, TR, 1, 1, 2, 2, 2, 4, 64, false, false)           \
  WHAT(LINKAGE, PREFIX##any_32x32, TR, 1, 1, 1, 1, 4, 4, 64, false, false)
#define ASC_TILE_KERNELS_F32(WHAT, LINKAGE, PREFIX, TR)                              \
  WHAT(LINKAGE, PREFIX##128x128, TR, 2, 1, 2, 4, 1, 4, 128, true, false)             \
  WHAT(LINKAGE, PREFIX##64x64, TR, 1, 1, 2, 2, 2, 4, 128, true, true)                \
  WHAT(LINKAGE, PREFIX##32x32, TR, 1, 1, 1, 1, 4, 5, 64, true, true)                 \
  WHAT(LINKAGE, PREFIX##any_128x128, TR, 2, 1, 2, 4, 1, 4, 64, false, false)         \
  WHAT(LINKAGE, PREFIX##any_64x64, TR, 1, 1, 2, 2, 2, 4, 64, false, false)           \
  WHAT(LINKAGE, PREFIX##any_32x32, TR, 1, 1, 1, 1, 4, 4, 64, false, false)

// The kernels of each input type with one linkage and prefix.
#define ASC_TILE_KERNELS_BF16(WHAT, LINKAGE, PREFIX) \
  ASC_TILE_KERNELS_MFMA(WHAT, LINKAGE, PREFIX##bf16_, asc::tile::Tr16<true>)
#define ASC_TILE_KERNELS_F16(WHAT, LINKAGE, PREFIX) \
  ASC_TILE_KERNELS_MFMA(WHAT, LINKAGE, PREFIX##f16_, asc::tile::Tr16<false>)
#define ASC_TILE_KERNELS_FP32(WHAT, LINKAGE, PREFIX) \
  ASC_TILE_KERNELS_F32(WHAT, LINKAGE, PREFIX##f32_, asc::tile::TrF32)
#define ASC_TILE_KERNELS_I8(WHAT, LINKAGE, PREFIX) \
  ASC_TILE_KERNELS_MFMA(WHAT, LINKAGE, PREFIX##i8_, asc::tile::TrI8)
// Host tables in variant order (after the kernels' declarations).
#define ASC_TILE_TABLE_MFMA(PREFIX)                                                                          \
  {PREFIX##256x256, PREFIX##128x256, PREFIX##192x128, PREFIX##128x128, PREFIX##64x64, PREFIX##64x64k2,       \
   PREFIX##32x64, PREFIX##32x32, PREFIX##any_256x256, PREFIX##any_128x128, PREFIX##any_64x64, PREFIX##any_32x32}
#define ASC_TILE_TABLE_F32(PREFIX) \
  {PREFIX##128x128, PREFIX##64x64, PREFIX##32x32, PREFIX##any_128x128, PREFIX##any_64x64, PREFIX##any_32x32}
