// MFMA GEMM on small and ragged tiles for gfx950: the shapes that the 256x256 tiles of
// gemm_direct.h cannot take (a dimension that is no multiple of the tile, an operand that
// is not 16-byte aligned) or leave most of the chip idle (few output tiles).
//
//   - A workgroup owns a kBM x kBN output tile.  Its waves form kKW groups of kWM x kWN
//     waves; a group computes the whole tile over its own share of K (k-tiles g, g + kKW,
//     ...), each wave kI x kJ blocks of 32x32 MFMA accumulators, and the groups' partial
//     tiles are summed through LDS in group order.  Splitting K inside the workgroup keeps
//     all four SIMDs busy on tiles too small to split further in M and N, without a
//     workspace and with a fixed summation order.
//   - A k-tile is kKB = 64 or 128 bytes of K, in k-steps of one 16-byte chunk per lane half.
//     128 bytes fetch whole L2 lines of A's rows; 64 bytes leave room for more stages.
//   - kDma (operands 16-byte aligned, row strides and K, N whole 16-byte chunks): operands
//     go from memory straight into kStages LDS stages (buffer_load ... lds).  The buffer
//     descriptors end where the operand ends, so rows of A past M and rows of B past K read
//     as zero; chunks of A past K are sent out of bounds lane by lane; columns of B past N
//     only reach columns of C that are not stored.  With kLean a k-tile is waited for when
//     its iteration starts (kStages - 1 tiles in flight); without, its first operands are
//     read an iteration early (kStages - 2 in flight), which pays when the MFMAs are the
//     bound.
//   - otherwise: 16-byte global loads at element alignment into kSets register sets (that
//     many k-tiles in flight), then into two LDS stages; rows are clamped, the last k-tile
//     is loaded with element checks.
//   - LDS tiles: A rows of kKB bytes, B rows as in memory (N contiguous), both with 16-byte
//     chunks swizzled per row so that one pass of an operand read covers all banks.
//
// What bounds the tiles (fp16/bf16, gfx950): operand traffic from the L2 per MFMA cycle is
// 32 bytes per CU and clock for 256x256, 48 for 128x256, 64 for 128x128, 128 for 64x64, of
// the 64 the L1 path delivers, so a larger tile wins as soon as its tiles fill the CUs;
// short problems are bound by the chain of load latencies, so small tiles split K over
// the waves and keep up to 128 KiB of loads in flight per CU.
#pragma once

#include <utility>

#include "gemm_common.h"
#include "numeric.h"

namespace asc {
namespace gemm {

typedef short tile_i16x4 __attribute__((ext_vector_type(4)));
typedef int tile_i32x2 __attribute__((vector_size(8)));

enum TileOut { kTileOutF32 = 0, kTileOutF16 = 1, kTileOutBF16 = 2, kTileOutI32 = 3 };

// A vector stored or loaded at the alignment of its elements.
template <class V, class E>
struct __attribute__((packed, aligned(alignof(E)))) ElemAligned {
  V v;
};

// The arguments of every tile kernel.
struct TileArgs {
  const void* a;
  const void* b;
  void* c;
  const float* vec;  // fp32 per column: the bias (or null), int8: the dequant scale
  int64_t lda, ldb, ldc;  // elements
  int M, N, K;
  int tiles_m, tiles_n;
  int out;     // TileOut
  int act;     // 0 none, 1 relu, 2 leaky relu (float kernels)
  float alpha;
  int trunc19;  // int8: clear the low 13 mantissa bits of the scale
  int reserved;  // the struct is its own size as an argument blob: no padding after it
};
static_assert(sizeof(TileArgs) == 96, "argument blob");

// Logical tile of a workgroup: consecutive logical ids live on one XCD (workgroup b runs on
// XCD b % 8), and kGroup tile rows are walked together so that A and B panels stay in its L2.
__device__ __forceinline__ void tile_of_block(int bid, int nblocks, int tiles_m, int tiles_n, int group_m, int& tm,
                                              int& tn) {
  const int per = nblocks >> 3, extra = nblocks & 7, xcd = bid & 7;
  const int logical = xcd * per + min(xcd, extra) + (bid >> 3);
  const int group_size = group_m * tiles_n;
  const int group = logical / group_size;
  const int first_m = group * group_m;
  const int gm = min(tiles_m - first_m, group_m);
  const int in_group = logical - group * group_size;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}

template <class Tr, int kI_, int kJ_, int kWM_, int kWN_, int kKW_, int kStages_, int kKB_, bool kDma_, bool kLean_ = false>
struct TileGemm {
  using Elem = typename Tr::Elem;
  using Acc = typename Tr::Acc;
  static constexpr int kI = kI_, kJ = kJ_, kWM = kWM_, kWN = kWN_, kKW = kKW_;
  static constexpr bool kDma = kDma_, kLean = kLean_;
  static constexpr int kStages = kDma ? kStages_ : 2;  // LDS stages
  static constexpr int kSets = kStages_;               // register sets of the register path (k-tiles in flight)
  static constexpr int kES = sizeof(Elem);
  static constexpr int kKB = kKB_;        // bytes of K per k-tile
  static constexpr int kBK = kKB / kES;   // K elements per k-tile
  static constexpr int kSteps = kKB / 32;  // MFMA k-steps: one 16-byte chunk per lane half each
  static constexpr int kBM = 32 * kI * kWM, kBN = 32 * kJ * kWN;
  static constexpr int kGroupWaves = kWM * kWN;
  static constexpr int kWaves = kGroupWaves * kKW, kThreads = 64 * kWaves;
  static constexpr int kBOff = kBM * kKB;
  static constexpr int kStageBytes = kKB * (kBM + kBN);  // one group's stage
  static constexpr int kStageTotal = kStageBytes * kKW;
  static constexpr int kRowBytes = kBN * kES;  // one B row in LDS
  static constexpr int kLoadsA = kBM * kKB / 1024 / kGroupWaves, kLoadsB = kBN * kKB / 1024 / kGroupWaves;
  static constexpr int kLoads = kLoadsA + kLoadsB;  // 1 KiB loads per wave and k-tile
  // loads that may still run when a k-tile's iteration ends: those of the tiles beyond the next two
  static constexpr int kInFlight = kLoads * (kStages - (kLean ? 2 : 3));
  static constexpr int kOob = 0x7ffffff0;  // past every descriptor's end
  static_assert(kDma || kSets % 2 == 0, "the register ring is unrolled over two LDS stages");
  static_assert(!kDma || kStages >= 3, "the ring holds the tile read, the next one and those in flight");
  static_assert(kRowBytes <= 1024 && (kBN & (kBN - 1)) == 0, "a load covers whole rows of B");
  static_assert(kKB == 64 || kKB == 128, "A rows of 4 or 8 chunks");
  static_assert(kBM * kKB / 1024 % kGroupWaves == 0 && kBN * kKB / 1024 % kGroupWaves == 0, "whole loads per wave");
  // LDS bytes of a stage: at the end the ring holds the groups' partial tiles
  static constexpr int kPartials = kKW == 1 ? 0 : kWaves * kI * kJ * 4096;
  static constexpr int kLdsStage =
      kStageTotal * kStages >= kPartials ? kStageTotal : (kPartials / kStages + 1023) / 1024 * 1024;

  // A chunk swizzle: the 16 rows that one pass of a b128 read covers get distinct 16-byte
  // parts of the 256-byte bank line.
  __device__ __forceinline__ static int a_swz(int row) { return kKB == 64 ? (row >> 2) & 3 : (row >> 1) & 7; }
  // B chunk swizzle: position p of row r holds logical chunk p ^ b_swz(r).  A transpose read
  // covers 4 rows x 64 bytes (16-bit) or 8 rows x 32 bytes (8-bit) per 32 lanes, an fp32 read
  // rows r and r + 4 x 128 bytes: the swizzle gives those rows distinct 64-, 32- or 128-byte
  // parts of the 256-byte bank line.
  __device__ __forceinline__ static int b_swz(int row) {
    if constexpr (kES == 2) {
      if constexpr (kRowBytes >= 256) return (0xCA60u >> (4 * (row & 3))) & 15;
      else if constexpr (kRowBytes == 128) return ((row >> 1) & 1) << 2;
      else return 0;
    } else if constexpr (kES == 1) {
      if constexpr (kRowBytes >= 256) return (0xE5CB2097u >> (4 * (row & 7))) & 15;
      else if constexpr (kRowBytes == 128) return ((row >> 1) & 3) << 1;
      else if constexpr (kRowBytes == 64) return ((row >> 2) & 1) << 1;
      else return 0;
    } else {
      if constexpr (kRowBytes >= 256) return ((row >> 2) & 1) << 3;
      else return 0;
    }
  }

  const uint8_t* a;  // row m0 of A
  const uint8_t* b;  // column n0 of B
  int lane, gw, kw, wm, wn;  // wave in its group, group, the wave's place in the tile
  int k_bytes, K, rows, cols;  // of A's rows: bytes; K; rows and columns of the tile inside C
  int64_t lda_b, ldb_b;        // bytes
  uint8_t* lds[kStages];       // this group's part of each stage

  // ---- direct-to-LDS loads
  int voff_a[kLoadsA], voff_b[kLoadsB];
  int a_total, b_cols;
  __amdgpu_buffer_rsrc_t ra, rb;  // of the k-tile last issued

  // Lane's row and logical chunk of its i-th A / B load.
  static constexpr int kChunks = kKB / 16;  // of a row of A
  __device__ __forceinline__ int a_row(int i) const { return 64 / kChunks * (gw * kLoadsA + i) + lane / kChunks; }
  __device__ __forceinline__ int a_byte(int i) const { return ((lane % kChunks) ^ a_swz(a_row(i))) * 16; }
  static constexpr int kLanesPerRow = kRowBytes / 16;
  static constexpr int kRowsPerLoad = 64 / kLanesPerRow;
  __device__ __forceinline__ int b_row(int i) const {
    return kRowsPerLoad * (gw * kLoadsB + i) + lane / kLanesPerRow;
  }
  __device__ __forceinline__ int b_byte(int i) const { return ((lane % kLanesPerRow) ^ b_swz(b_row(i))) * 16; }

  __device__ __forceinline__ void init_dma() {
    const int lda = static_cast<int>(lda_b), ldb = static_cast<int>(ldb_b);
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) voff_a[i] = a_row(i) * lda + a_byte(i);
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) voff_b[i] = b_row(i) * ldb + b_byte(i);
    a_total = (min(rows, kBM) - 1) * lda + k_bytes;
    b_cols = min(cols, kBN) * kES;
  }

  // Descriptors of k-tile kt: each operand's starts at the k-tile and ends with the operand.
  __device__ __forceinline__ void set_descriptors(int kt) {
    ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a + static_cast<int64_t>(kt) * kKB),
                                           static_cast<short>(0), max(a_total - kt * kKB, 0), 0x00020000);
    const int krows = min(K - kt * kBK, kBK);
    rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(b + static_cast<int64_t>(kt) * kBK * ldb_b),
                                           static_cast<short>(0),
                                           krows > 0 ? (krows - 1) * static_cast<int>(ldb_b) + b_cols : 0, 0x00020000);
  }

  // k-tile kt (past the last one: zeros, without memory traffic) into stage kS.
  template <int kS>
  __device__ __forceinline__ void issue(int kt) {
    set_descriptors(kt);
    const int left = k_bytes - kt * kKB;  // bytes of a row of A from here on
    uint8_t* base = lds[kS];
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, (__attribute__((address_space(3))) void*)(base + (gw * kLoadsA + i) * 1024), 16,
          a_byte(i) < left ? voff_a[i] : kOob, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rb, (__attribute__((address_space(3))) void*)(base + kBOff + (gw * kLoadsB + i) * 1024), 16, voff_b[i], 0,
          0, 0);
    }
  }

  // ---- loads through registers
  struct Regs {
    u32x4 a[kLoadsA], b[kLoadsB];
  };
  // 16 bytes at element alignment
  __device__ __forceinline__ static u32x4 load16(const uint8_t* p) {
    return reinterpret_cast<const ElemAligned<u32x4, Elem>*>(p)->v;
  }
  // The first n (0..16/kES) elements at p, zeros behind them.
  __device__ __forceinline__ static u32x4 load_part(const uint8_t* p, int n) {
    if (n * kES >= 16) return load16(p);
    Elem e[16 / kES];
#pragma unroll
    for (int i = 0; i < 16 / kES; ++i) e[i] = i < n ? reinterpret_cast<const Elem*>(p)[i] : Elem(0);
    u32x4 v;
    __builtin_memcpy(&v, e, 16);
    return v;
  }

  __device__ __forceinline__ void fetch(int kt, int k_tiles, Regs& r) const {
    // Every chunk of a k-tile before the last lies inside its row of A; its rows of B are
    // followed by another row at least 16 bytes long (ldb_b >= 16 here, else every tile is
    // loaded with checks), so a chunk that runs past N stays inside the matrix.
    if (kt < k_tiles - 1 && ldb_b >= 16) {
      const uint8_t* at = a + static_cast<int64_t>(kt) * kKB;
#pragma unroll
      for (int i = 0; i < kLoadsA; ++i) r.a[i] = load16(at + min(a_row(i), rows - 1) * lda_b + a_byte(i));
      const uint8_t* bt = b + static_cast<int64_t>(kt) * kBK * ldb_b;
#pragma unroll
      for (int i = 0; i < kLoadsB; ++i) {
        const int cb = b_byte(i) < cols * kES ? b_byte(i) : 0;
        r.b[i] = load16(bt + b_row(i) * ldb_b + cb);
      }
      return;
    }
    const int k0 = kt * kBK;
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) {
      const int e = a_byte(i) / kES;
      const int n = a_row(i) < rows ? K - k0 - e : 0;
      r.a[i] = n > 0 ? load_part(a + a_row(i) * lda_b + static_cast<int64_t>(k0 + e) * kES, n) : u32x4{};
    }
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) {
      const int e = b_byte(i) / kES;
      const int n = k0 + b_row(i) < K ? cols - e : 0;
      r.b[i] = n > 0 ? load_part(b + static_cast<int64_t>(k0 + b_row(i)) * ldb_b + static_cast<int64_t>(e) * kES, n)
                     : u32x4{};
    }
  }

  template <int kS>
  __device__ __forceinline__ void stash(const Regs& r) {
    uint8_t* base = lds[kS] + lane * 16;
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) *reinterpret_cast<u32x4*>(base + (gw * kLoadsA + i) * 1024) = r.a[i];
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) *reinterpret_cast<u32x4*>(base + kBOff + (gw * kLoadsB + i) * 1024) = r.b[i];
  }

  // ---- operands of k-step `step` (0 .. kSteps - 1) from stage kS
  __device__ __forceinline__ static int b_off(int row, int col) {
    const int byte = col * kES;
    return row * kRowBytes + (((byte >> 4) ^ b_swz(row)) << 4) + (byte & 15);
  }

  template <int kS>
  __device__ __forceinline__ void read_frags(int step, u32x4 (&fa)[kI], u32x4 (&fb)[kJ]) const {
    const uint8_t* as = lds[kS];
    const uint8_t* bs = as + kBOff;
    const int h = lane >> 5;
    const int chunk = step * 2 + h;
    const int arow = wm * (32 * kI) + (lane & 31);
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int row = arow + i * 32;
      fa[i] = *reinterpret_cast<const u32x4*>(as + row * kKB + ((chunk ^ a_swz(row)) << 4));
    }
    const int g = (lane >> 4) & 1, t = lane & 15;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      const int nb = wn * (32 * kJ) + j * 32;
      if constexpr (kES == 2) {
        // k = 16*step + 8h + e; read e = 0..3 then 4..7; lane 4jj+q -> row +jj, col +4q
        const int row = step * 16 + 8 * h + (t >> 2);
        const int col = nb + 16 * g + 4 * (t & 3);
        const tile_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tile_i16x4*)(bs + b_off(row, col)));
        const tile_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tile_i16x4*)(bs + b_off(row + 4, col)));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        fb[j] = u32x4{l2[0], l2[1], h2[0], h2[1]};
      } else if constexpr (kES == 1) {
        // k = 32*step + 16h + e; read e = 0..7 then 8..15; lane 2jj+sub -> row +jj, col +8sub
        const int row = step * 32 + 16 * h + (t >> 1);
        const int col = nb + 16 * g + 8 * (t & 1);
        const tile_i32x2 lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (__attribute__((address_space(3))) tile_i32x2*)(bs + b_off(row, col)));
        const tile_i32x2 hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (__attribute__((address_space(3))) tile_i32x2*)(bs + b_off(row + 8, col)));
        fb[j] = u32x4{static_cast<uint32_t>(lo[0]), static_cast<uint32_t>(lo[1]), static_cast<uint32_t>(hi[0]),
                      static_cast<uint32_t>(hi[1])};
      } else {
        // k = 4*chunk + e in A and B alike: the four MFMAs of a chunk cover its four k
#pragma unroll
        for (int e = 0; e < 4; ++e)
          fb[j][e] = *reinterpret_cast<const uint32_t*>(bs + b_off(4 * chunk + e, nb + (lane & 31)));
      }
    }
  }

  __device__ __forceinline__ static void mma(Acc (&acc)[kI][kJ], const u32x4 (&fa)[kI], const u32x4 (&fb)[kJ]) {
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
      for (int j = 0; j < kJ; ++j) acc[i][j] = Tr::mfma(fa[i], fb[j], acc[i][j]);
  }

  // Meets the group's other waves; does not wait for outstanding loads.
  __device__ __forceinline__ static void group_barrier() {
    if constexpr (kGroupWaves > 1) asm volatile("s_barrier" ::: "memory");
  }

  // Iteration t of this group (k-tile kw + kKW * t, in stage kS).  On entry its k-step-0
  // operands are in fa0/fb0 and the k-tiles of iterations t and t+1 are visible in LDS.
  template <int kS>
  __device__ __forceinline__ void iteration(int t, Acc (&acc)[kI][kJ], u32x4 (&fa0)[kI], u32x4 (&fb0)[kJ],
                                            u32x4 (&fa1)[kI], u32x4 (&fb1)[kJ]) {
    constexpr int kNext = (kS + 1) % kStages, kAhead = (kS + kStages - 1) % kStages;
    if constexpr (kLean) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(kInFlight) : "memory");
      group_barrier();
      issue<kAhead>(kw + kKW * (t + kStages - 1));
      read_frags<kS>(0, fa0, fb0);
#pragma unroll
      for (int s = 0; s < kSteps; s += 2) {
        read_frags<kS>(s + 1, fa1, fb1);
        mma(acc, fa0, fb0);
        if (s + 2 < kSteps) read_frags<kS>(s + 2, fa0, fb0);
        mma(acc, fa1, fb1);
      }
      return;
    }
    issue<kAhead>(kw + kKW * (t + kStages - 1));
#pragma unroll
    for (int s = 0; s < kSteps; s += 2) {
      read_frags<kS>(s + 1, fa1, fb1);
      mma(acc, fa0, fb0);
      if (s + 2 < kSteps) read_frags<kS>(s + 2, fa0, fb0);
      else read_frags<kNext>(0, fa0, fb0);
      mma(acc, fa1, fb1);
    }
    // own loads of iteration t+2 done, and the reads of stage kS before it is refilled
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(kInFlight) : "memory");
    group_barrier();
  }
  template <int... kS>
  __device__ __forceinline__ void ring(std::integer_sequence<int, kS...>, int t, int n, Acc (&acc)[kI][kJ],
                                       u32x4 (&fa0)[kI], u32x4 (&fb0)[kJ], u32x4 (&fa1)[kI], u32x4 (&fb1)[kJ]) {
    ((t + kS < n ? iteration<kS>(t + kS, acc, fa0, fb0, fa1, fb1) : void()), ...);
  }
  template <int... kS>
  __device__ __forceinline__ void prologue(std::integer_sequence<int, kS...>) {
    (issue<kS>(kw + kKW * kS), ...);
  }

  // Iteration t of the register path: stage t % 2 holds its k-tile, register set (t+1) % kSets
  // that of iteration t+1, which goes into the other stage here; the set is then requested
  // again for iteration t+1+kSets.
  template <int kU>
  __device__ __forceinline__ void reg_iteration(int t, int k_tiles, Acc (&acc)[kI][kJ], Regs (&sets)[kSets]) {
    constexpr int kS = kU & 1, kSet = (kU + 1) % kSets;
    stash<kS ^ 1>(sets[kSet]);
    fetch(kw + kKW * (t + 1 + kSets), k_tiles, sets[kSet]);
    u32x4 fa0[kI], fb0[kJ], fa1[kI], fb1[kJ];
    read_frags<kS>(0, fa0, fb0);
#pragma unroll
    for (int s = 0; s < kSteps; s += 2) {
      read_frags<kS>(s + 1, fa1, fb1);
      mma(acc, fa0, fb0);
      if (s + 2 < kSteps) read_frags<kS>(s + 2, fa0, fb0);
      mma(acc, fa1, fb1);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    group_barrier();
  }
  template <int... kU>
  __device__ __forceinline__ void reg_ring(std::integer_sequence<int, kU...>, int t, int n, int k_tiles,
                                           Acc (&acc)[kI][kJ], Regs (&sets)[kSets]) {
    ((t + kU < n ? reg_iteration<kU>(t + kU, k_tiles, acc, sets) : void()), ...);
  }

  __device__ __forceinline__ void run(Acc (&acc)[kI][kJ]) {
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
      for (int j = 0; j < kJ; ++j) acc[i][j] = Acc{};
    const int k_tiles = (K + kBK - 1) / kBK;
    const int n = (k_tiles + kKW - 1) / kKW;  // iterations, alike in every group
    if constexpr (kDma) {
      init_dma();
      prologue(std::make_integer_sequence<int, kStages - 1>());
      u32x4 fa0[kI], fb0[kJ], fa1[kI], fb1[kJ];
      if constexpr (!kLean) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kInFlight) : "memory");
        group_barrier();
        read_frags<0>(0, fa0, fb0);
      }
      for (int t = 0; t < n; t += kStages)
        ring(std::make_integer_sequence<int, kStages>(), t, n, acc, fa0, fb0, fa1, fb1);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may outlive the loop
    } else {
      Regs sets[kSets];
#pragma unroll
      for (int u = 0; u < kSets; ++u) fetch(kw + kKW * u, k_tiles, sets[u]);
      stash<0>(sets[0]);
      fetch(kw + kKW * kSets, k_tiles, sets[0]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      group_barrier();
      for (int t = 0; t < n; t += kSets)
        reg_ring(std::make_integer_sequence<int, kSets>(), t, n, k_tiles, acc, sets);
    }
  }
};

// The output tile of one workgroup.  Tr::out_bits(value, vec_n, args) turns an accumulator
// value of column n into the output's bits.
template <class T, class Tr>
__device__ __forceinline__ void tile_body(const TileArgs& p) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the kernels' launch stubs
  constexpr int kS = T::kStages;
  // the LDS stages as distinct objects, so that the compiler can tell that loads into one
  // do not alias reads of another
  __shared__ __attribute__((aligned(16))) uint8_t lds0[T::kLdsStage];
  __shared__ __attribute__((aligned(16))) uint8_t lds1[T::kLdsStage];
  __shared__ __attribute__((aligned(16))) uint8_t lds2[kS > 2 ? T::kLdsStage : 16];
  __shared__ __attribute__((aligned(16))) uint8_t lds3[kS > 3 ? T::kLdsStage : 16];
  __shared__ __attribute__((aligned(16))) uint8_t lds4[kS > 4 ? T::kLdsStage : 16];
  static_assert(kS <= 5, "one __shared__ stage object per ring stage");
  uint8_t* const stages[5] = {lds0, lds1, lds2, lds3, lds4};
  int tm, tn;
  tile_of_block(blockIdx.x, p.tiles_m * p.tiles_n, p.tiles_m, p.tiles_n, 8, tm, tn);
  const int m0 = tm * T::kBM, n0 = tn * T::kBN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  T L;
  L.lane = lane;
  L.kw = wave / T::kGroupWaves;
  L.gw = wave % T::kGroupWaves;
  L.wm = L.gw / T::kWN;
  L.wn = L.gw % T::kWN;
  L.lda_b = p.lda * T::kES;
  L.ldb_b = p.ldb * T::kES;
  L.a = static_cast<const uint8_t*>(p.a) + m0 * L.lda_b;
  L.b = static_cast<const uint8_t*>(p.b) + static_cast<int64_t>(n0) * T::kES;
  L.K = p.K;
  L.k_bytes = p.K * T::kES;
  L.rows = p.M - m0;
  L.cols = p.N - n0;
#pragma unroll
  for (int s = 0; s < kS; ++s) L.lds[s] = stages[s] + L.kw * T::kStageBytes;
  typename T::Acc acc[T::kI][T::kJ];
  L.run(acc);

  // Epilogue.  MFMA 32x32 result layout: lane l holds column l%32 of a block, register r row
  // 8*(r/4) + 4*(l/32) + r%4.  A group of four registers is transposed across its quad of
  // lanes so that a lane stores four consecutive columns of one row.
  const int t = lane & 3, q = (lane & 31) >> 2, h = lane >> 5;
  const int mb = m0 + L.wm * 32 * T::kI, nb = n0 + L.wn * 32 * T::kJ;
  float vec_n[T::kJ];
#pragma unroll
  for (int j = 0; j < T::kJ; ++j) {
    const int n = nb + j * 32 + (lane & 31);
    vec_n[j] = n < p.N ? Tr::vec_at(p, n) : 0.0f;
  }
  constexpr int kUnits = T::kI * T::kJ * 4;
  constexpr int kPerStage = T::kLdsStage / 1024;
  // Partial tiles go through the ring (free now): unit u = 1 KiB = one register group of one
  // block of one wave; the groups' waves of one place then sum every kKW-th unit each.
  const auto unit = [&](int group, int u) -> uint8_t* {
    const int at = (L.gw * T::kKW + group) * kUnits + u;
    uint8_t* base = lds0;
    const int s = at / kPerStage;
    if constexpr (kS > 1) base = s == 1 ? lds1 : base;
    if constexpr (kS > 2) base = s == 2 ? lds2 : base;
    if constexpr (kS > 3) base = s == 3 ? lds3 : base;
    if constexpr (kS > 4) base = s == 4 ? lds4 : base;
    return base + (at - s * kPerStage) * 1024 + lane * 16;
  };
  if constexpr (T::kKW > 1) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < T::kI; ++i)
#pragma unroll
      for (int j = 0; j < T::kJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const typename Tr::Val x[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                                         acc[i][j][4 * g + 3]};
          u32x4 bits;
          __builtin_memcpy(&bits, x, 16);
          *reinterpret_cast<u32x4*>(unit(L.kw, (i * T::kJ + j) * 4 + g)) = bits;
        }
    __syncthreads();
  }
  // kEdge: the tile's last columns lie past N (element stores); otherwise four columns go
  // out in one store at element alignment, rows past M masked.
  const auto store = [&](auto edge, auto out_c, int i, int j, int g, const typename Tr::Val (&x)[4], float vn) {
    constexpr bool kEdge = decltype(edge)::value;
    constexpr int kOut = decltype(out_c)::value;
    const int row = mb + i * 32 + g * 8 + h * 4 + t, col = nb + j * 32 + 4 * q;
    uint32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = Tr::template out_bits<kOut>(x[e], vn, p);
    const int64_t off = row * p.ldc + col;
    if constexpr (kOut == kTileOutF32 || kOut == kTileOutI32) {
      quad_transpose_b32(v, t);
      if (row >= p.M) return;
      uint32_t* c = static_cast<uint32_t*>(p.c) + off;
      if constexpr (kEdge) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < p.N) c[e] = v[e];
      } else {
        reinterpret_cast<ElemAligned<u32x4, uint32_t>*>(c)->v = u32x4{v[0], v[1], v[2], v[3]};
      }
    } else {
      uint32_t d0 = (v[0] & 0xFFFFu) | (v[1] << 16), d1 = (v[2] & 0xFFFFu) | (v[3] << 16);
      quad_transpose_b16(d0, d1, t);
      if (row >= p.M) return;
      uint16_t* c = static_cast<uint16_t*>(p.c) + off;
      if constexpr (kEdge) {
        if (col < p.N) c[0] = static_cast<uint16_t>(d0);
        if (col + 1 < p.N) c[1] = static_cast<uint16_t>(d0 >> 16);
        if (col + 2 < p.N) c[2] = static_cast<uint16_t>(d1);
        if (col + 3 < p.N) c[3] = static_cast<uint16_t>(d1 >> 16);
      } else {
        reinterpret_cast<ElemAligned<u32x2, uint16_t>*>(c)->v = u32x2{d0, d1};
      }
    }
  };
  const auto finish = [&](auto edge, auto out_c) {
  if constexpr (T::kKW == 1) {
#pragma unroll
    for (int i = 0; i < T::kI; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < T::kJ; ++j) {
          const typename Tr::Val x[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                                         acc[i][j][4 * g + 3]};
          store(edge, out_c, i, j, g, x, vec_n[j]);
        }
  } else {
#pragma unroll
    for (int k = 0; k < (kUnits + T::kKW - 1) / T::kKW; ++k) {
      const int u = k * T::kKW + L.kw;
      if (u < kUnits) {
        typename Tr::Val x[4] = {};
#pragma unroll
        for (int group = 0; group < T::kKW; ++group) {
          const u32x4 bits = *reinterpret_cast<const u32x4*>(unit(group, u));
          typename Tr::Val y[4];
          __builtin_memcpy(y, &bits, 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = group == 0 ? y[e] : x[e] + y[e];
        }
        const int blk = u >> 2;
        float vn = vec_n[0];
#pragma unroll
        for (int j = 1; j < T::kJ; ++j) vn = blk % T::kJ == j ? vec_n[j] : vn;
        store(edge, out_c, blk / T::kJ, blk % T::kJ, u & 3, x, vn);
      }
    }
  }
  };
  const auto by_out = [&](auto edge) {
    if constexpr (Tr::kInt) {
      if (p.out == kTileOutI32) finish(edge, std::integral_constant<int, kTileOutI32>());
      else finish(edge, std::integral_constant<int, kTileOutF16>());
    } else {
      if (p.out == kTileOutF32) finish(edge, std::integral_constant<int, kTileOutF32>());
      else if (p.out == kTileOutF16) finish(edge, std::integral_constant<int, kTileOutF16>());
      else finish(edge, std::integral_constant<int, kTileOutBF16>());
    }
  };
  if (n0 + T::kBN <= p.N) by_out(std::false_type());
  else by_out(std::true_type());
#endif

}

}  // namespace gemm
}  // namespace asc
