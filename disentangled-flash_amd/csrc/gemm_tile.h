// Tile configurations of the projection GEMM (gemm.hip) and the addresses its copies
// read, apart from the kernel: plain constexpr functions, so that a host program can check
// for every configuration, split and K that no copy leaves its operand.
#pragma once

#include <stdint.h>

namespace dflash {

constexpr int kStepK = 32;           // k of one MFMA step
constexpr int kSlabK = 2 * kStepK;    // k of one slab (128-byte rows)

// Chunk permutation of slab row r: 16-byte chunk k of the row sits at position
// k ^ slab_swizzle(r).  Eight consecutive rows hit eight different chunks of a
// 128-byte window, and of sixteen no two the same chunk of a 256-byte one.
// Depends on r mod 16 only.
constexpr int slab_swizzle(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Output column (inside the tile) of W row r of a slab: row x = 4a + b of the
// 16-row blocks 2i and 2i + 1 holds columns 32i + 8a + b and 32i + 8a + 4 + b.
constexpr int w_row(int r) {
  const int block = r >> 4;
  const int x = r & 15;
  return 8 * (x >> 2) + (x & 3) + 4 * (block & 1) + 32 * (block >> 1);
}

// Tile configuration: a workgroup of WAVES_M x WAVES_N wavefronts computes a
// BM x BN tile of Y (wavefront tile BM/WAVES_M x BN/WAVES_N) through a ring of
// STAGES slabs; WGS workgroups per CU are budgeted for.
template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int WGS_, int STAGES_ = 2>
struct GemmConfig {
  static constexpr int BM = BM_;
  static constexpr int BN = BN_;
  static constexpr int WAVES_M = WAVES_M_;
  static constexpr int WAVES_N = WAVES_N_;
  static constexpr int WGS = WGS_;
  static constexpr int STAGES = STAGES_;
  static constexpr int WAVES = WAVES_M * WAVES_N;
  static constexpr int THREADS = 64 * WAVES;
  static constexpr int WM = BM / WAVES_M;
  static constexpr int WN = BN / WAVES_N;
  static constexpr int MB = WM / 16;            // 16-row blocks per wavefront
  static constexpr int NB = WN / 16;            // 16-column blocks per wavefront
  static constexpr int A_LOADS = BM / 8 / WAVES;  // copies (8 rows each) per wavefront and slab
  static constexpr int B_LOADS = BN / 8 / WAVES;
  static constexpr int LOADS = A_LOADS + B_LOADS;
  static constexpr int A_BYTES = BM * kSlabK * 2;
  static constexpr int SLAB = (BM + BN) * kSlabK * 2;
  static constexpr int LDS = STAGES * SLAB;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "copies split evenly");
  static_assert(WM % 16 == 0 && WN % 32 == 0, "whole MFMA blocks, column blocks in pairs");
  static_assert(STAGES >= 2 && LDS * WGS <= 160 * 1024, "LDS of a CU");
  static_assert((STAGES - 1) * LOADS <= 63, "vmcnt range");
};

// Columns are a multiple of the tile's, rows ragged.  Large tiles need the fewest bytes per
// product and fill the chip from about 256 tiles; small ones, with deeper rings, give few
// rows more workgroups.
using Cfg128x192 = GemmConfig<128, 192, 2, 2, 2>;
using Cfg128x128 = GemmConfig<128, 128, 2, 2, 2>;
using Cfg256x192 = GemmConfig<256, 192, 4, 2, 1>;
using Cfg64x128 = GemmConfig<64, 128, 2, 2, 2, 3>;
using Cfg64x64 = GemmConfig<64, 64, 2, 2, 4>;
using Cfg256x256 = GemmConfig<256, 256, 4, 2, 1>;
using Cfg128x192Deep = GemmConfig<128, 192, 4, 2, 1, 4>;
using Cfg128x128Deep = GemmConfig<128, 128, 4, 2, 1, 5>;
using Cfg128x64 = GemmConfig<128, 64, 4, 1, 2, 3>;
using Cfg64x64Deep = GemmConfig<64, 64, 2, 2, 2, 5>;
using Cfg32x64 = GemmConfig<32, 64, 2, 2, 2, 6>;

// The slabs of range `split` of `splits` of K (the last slab may be half: K % 32 == 0).
struct KRange {
  int first;  // slab
  int slabs;
  int k;      // from the range's first k to its last
};
constexpr KRange k_range(int K, int split, int splits) {
  const int all = (K + kSlabK - 1) / kSlabK;
  const int first = all * split / splits;
  const int slabs = all * (split + 1) / splits - first;
  const int rest = K - first * kSlabK;
  return {first, slabs, rest < slabs * kSlabK ? rest : slabs * kSlabK};
}

// The slab at place `kt` of an order that starts at slab `k0` of `slabs` and wraps around.
constexpr int slab_at(int kt, int k0, int slabs) { return kt + k0 < slabs ? kt + k0 : kt + k0 - slabs; }

// Copy j of a slab fetches eight slab rows, 16 bytes a lane: row and source chunk of a lane.
template <typename CF>
constexpr int copy_row(int j, int wave, int lane) {
  return (j * CF::WAVES + wave) * 8 + (lane >> 3);
}
constexpr int copy_chunk(int row, int lane) { return (lane & 7) ^ slab_swizzle(row); }

// Bytes of an operand's tile from the first k of a range in its first row to the end of its
// last row (row_bytes = 2 K of the whole operand).
constexpr uint32_t tile_bytes(int rows, uint32_t row_bytes, const KRange& range) {
  return static_cast<uint32_t>(rows) * row_bytes - static_cast<uint32_t>(range.first) * (kSlabK * 2);
}

// How the kernel addresses its copies: 32-bit offsets into a buffer resource, for K of
// whole slabs or with a half slab at its end, or 64-bit addresses.
enum class Copies { kWhole, kHalf, kFar };

// Where the copies of a slab read: from the tile's first row, 16 bytes at `lane` + `scalar`
// (the instruction's two offsets) of a buffer resource of `bytes`.  A raw buffer's range
// check is documented to compare `lane` alone with the size; the MI355X was seen to
// compare the sum.  Nothing may be read past the operand by either rule, and nothing needed
// be cut off:
//   * rows past the tile's last one are past `bytes` by `lane` alone;
//   * whole slabs end with their rows, so their place can be the scalar offset, which costs
//     no arithmetic per lane;
//   * of a half slab the last row's chunks past K lie past the operand (those of the rows
//     before are in the next row; their products are not computed), so its place goes into
//     the lane's offset.  (A resource that begins at the slab costs whole slabs twelve scalar
//     operations each: layers of 768 and 1536 columns 1.5-2.5 % slower.)
//   * places past the last slab read nothing: size 0.
struct SlabCopy {
  uint32_t lane, scalar, bytes;
};
template <Copies COPIES>
constexpr SlabCopy slab_copy(int kt, int k0, int slabs, uint32_t tile, uint32_t lane) {
  const uint32_t start = static_cast<uint32_t>(slab_at(kt, k0, slabs)) * (kSlabK * 2);
  const uint32_t bytes = kt < slabs ? tile : 0u;
  if (COPIES == Copies::kHalf) return {lane + start, 0u, bytes};
  return {lane, start, bytes};
}

// With 64-bit addresses (tile rows past 32-bit offsets): the k of a lane's chunk, where slabs
// and chunks past K repeat k of the last 8 (their products are not computed).
constexpr int far_k(int kt, int k0, const KRange& range, int chunk) {
  const int last = kt < range.slabs ? kt : range.slabs - 1;
  const int k = slab_at(last, k0, range.slabs) * kSlabK + chunk * 8;
  return k < range.k - 8 ? k : range.k - 8;
}

}  // namespace dflash
