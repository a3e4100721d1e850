"""No copy of the projection GEMM leaves its operand (CPU: the address functions of
``gemm_tile.h`` compiled for the host).

For every tile configuration, K around whole and half slabs, every split of K, every starting
slab of the k order and tiles of one, some and all rows, each copy of each lane is followed to the
bytes that it reads, under both rules that the range check of a raw buffer may follow (the lane's
offset alone, as documented, or the sum with the scalar offset).  They have to lie in the tile's
rows, and every k of every row has to be fetched once.
"""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "disentangled-flash_amd" / "csrc"

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "gemm_tile.h"
using namespace dflash;

static int failures = 0;
static void fail(const char* what, int bm, int bn, int K, int split, int splits, int rows) {
  if (failures++ < 20)
    std::printf("%s: tile %d x %d, K %d, range %d of %d, %d rows\n", what, bm, bn, K, split, splits, rows);
}

// One operand of a tile: `rows` rows, LOADS copies a wavefront and slab.
template <typename CF, Copies COPIES, int LOADS, bool IS_X>
static void operand(int K, int split, int splits, int rows) {
  const KRange range = k_range(K, split, splits);
  const int64_t row_bytes = 2LL * K;
  const int64_t base0 = 2LL * range.first * kSlabK;  // of the range's first k in the first row
  const int64_t extent = rows * row_bytes;           // of the operand, from the tile's first row
  for (int start = 0; start < (range.k % kSlabK == 0 ? 8 : 1); ++start) {
    const int k0 = (start * range.slabs) >> 3;
    std::vector<int> fetched(static_cast<size_t>(rows) * range.k / 8, 0);
    for (int kt = 0; kt < range.slabs + CF::STAGES; ++kt) {
      for (int j = 0; j < LOADS; ++j)
        for (int wave = 0; wave < CF::WAVES; ++wave)
          for (int lane = 0; lane < 64; ++lane) {
            const int row = copy_row<CF>(j, wave, lane);
            const int chunk = copy_chunk(row, lane);
            const int r = IS_X ? row : w_row(row);
            const SlabCopy s = slab_copy<COPIES>(
                kt, k0, range.slabs, tile_bytes(rows, static_cast<uint32_t>(row_bytes), range),
                static_cast<uint32_t>(r * row_bytes + chunk * 16));
            const int64_t off = static_cast<int64_t>(s.lane) + s.scalar;  // from the range's first k
            const int f = far_k(kt, k0, range, chunk);
            if (f < 0 || f + 8 > range.k) fail("64-bit address", CF::BM, CF::BN, K, split, splits, rows);
            for (int word = 0; word < 4; ++word) {
              if (static_cast<int64_t>(s.lane) + 4 * word + 4 > s.bytes) continue;
              if (base0 + off + 4 * word + 4 > extent) fail("outside", CF::BM, CF::BN, K, split, splits, rows);
            }
            if (kt >= range.slabs) {
              if (s.bytes != 0) fail("past the last slab", CF::BM, CF::BN, K, split, splits, rows);
              continue;
            }
            const int k = slab_at(kt, k0, range.slabs) * kSlabK + chunk * 8;
            if (r >= rows || k >= range.k) continue;  // products not computed or not stored
            if (off + 16 > s.bytes || off != r * row_bytes + 2LL * k || f != k)
              fail("not fetched", CF::BM, CF::BN, K, split, splits, rows);
            fetched[static_cast<size_t>(r) * (range.k / 8) + k / 8]++;
          }
    }
    for (int n : fetched)
      if (n != 1) {
        fail("not once", CF::BM, CF::BN, K, split, splits, rows);
        break;
      }
  }
}

template <typename CF>
static void config() {
  for (int K : {32, 64, 96, 128, 160, 480, 768, 1056, 2080})
    for (int splits : {1, 2, 4, 8}) {
      if (splits > (K + kSlabK - 1) / kSlabK) continue;
      for (int split = 0; split < splits; ++split) {
        if (K % kSlabK == 0) {
          for (int rows : {1, 17, CF::BM - 1, CF::BM})
            operand<CF, Copies::kWhole, CF::A_LOADS, true>(K, split, splits, rows);
          operand<CF, Copies::kWhole, CF::B_LOADS, false>(K, split, splits, CF::BN);
        } else {
          for (int rows : {1, 17, CF::BM - 1, CF::BM})
            operand<CF, Copies::kHalf, CF::A_LOADS, true>(K, split, splits, rows);
          operand<CF, Copies::kHalf, CF::B_LOADS, false>(K, split, splits, CF::BN);
        }
      }
    }
}

int main() {
  config<Cfg128x192>(); config<Cfg128x128>(); config<Cfg256x192>(); config<Cfg64x128>();
  config<Cfg64x64>(); config<Cfg256x256>(); config<Cfg128x192Deep>(); config<Cfg128x128Deep>();
  config<Cfg128x64>(); config<Cfg64x64Deep>(); config<Cfg32x64>();
  // The longest rows of the 32-bit form: a tile of 256 rows ends within 32 bits.
  const int K = (1 << 23) - 32;
  const KRange range = k_range(K, 0, 1);
  if (tile_bytes(256, 2u * K, range) != 512LL * K) fail("32 bits", 256, 256, K, 0, 1, 256);
  const SlabCopy s = slab_copy<Copies::kHalf>(range.slabs - 1, 0, range.slabs, 512u * K, 510u * K + 48);
  if (s.lane != 512LL * K - 16) fail("32 bits", 256, 256, K, 0, 1, 256);
  std::printf("%d failures\n", failures);
  return failures != 0;
}
"""


def test_copies_stay_inside_their_operand(tmp_path):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("g++ not available")
    source = tmp_path / "addresses.cpp"
    source.write_text(PROGRAM)
    program = tmp_path / "addresses"
    built = subprocess.run([compiler, "-std=c++17", "-O2", "-I", str(CSRC), str(source), "-o",
                            str(program)], capture_output=True, text=True)
    assert built.returncode == 0, built.stderr
    ran = subprocess.run([str(program)], capture_output=True, text=True)
    assert ran.returncode == 0, ran.stdout
