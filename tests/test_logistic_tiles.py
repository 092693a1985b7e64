"""Reads of the design matrix by the float64 logistic passes, on the host.

The passes of ``logistic_common.h`` read a row-major X[N][D] straight into matrix
operands, whole 16-feature tiles at a time; ``logistic_tiles.h`` holds their widths
and limits.  Every lane's offset in every block, also of the blocks read past the
end, has to lie in the row that it stands for, and the elements that exist have
to come from their own place.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <algorithm>
#include "logistic_tiles.h"
using namespace gjx::logistic;

static long bad = 0;
static void read(const char* pass, int N, int D, int row, int feature, long off) {
  const int r = std::min(row, N - 1);
  const long lo = 8L * r * D, hi = lo + 8L * D;
  const bool in_row = off >= lo && off + 8 <= hi;
  const bool own = feature >= D || off == lo + 8L * feature;
  if ((!in_row || !own) && bad++ < 5)
    std::printf("%s N=%d D=%d row %d feature %d reads byte %ld of row [%ld, %ld)\n", pass, N, D, row, feature, off, lo, hi);
}

template <int MAXD>
static void check(int N, int D) {
  const int nblk = (N + 15) / 16;
  by_width<MAXD>(D, [&](auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    if (16 * NB > MAXD) std::printf("D=%d: %d tiles past the capacity\n", D, NB), ++bad;
    for (int blk = 0; blk < nblk + 8; ++blk) {
      const int b0 = std::min(blk, nblk - 1), n0 = 16 * b0;
      const long base = 8L * n0 * D;
      for (int g = 0; g < 4; ++g)
        for (int m = 0; m < 16; ++m) {
          // Gram pass: rows 4 j + g, features 16 b + m
          for (int j = 0; j < 4; ++j) {
            const int r = 4 * j + g;
            const uint32_t row = row_bytes(8u * (uint32_t)(r * D), n0, N, D);
            for (int b = 0; b < NB; ++b)
              read("gram", N, D, n0 + r, 16 * b + m,
                   base + row + (b < NB - 1 ? 8u * (uint32_t)(m + 16 * b) : last_tile_bytes(NB, m, D)));
          }
          // quadratic forms: row m, pairs of neighbours, the last tile by pairs when it is whole
          const uint32_t row = row_bytes(8u * (uint32_t)(m * D), n0, N, D);
          for (int s = 0; s < 4 * NB; s += 2)
            for (int e = 0; e < 2; ++e) {
              const int f = quad_feature(s + e, g);
              const bool pair = s < 4 * NB - 4 || D == 16 * NB;
              read("quad", N, D, n0 + m, f,
                   base + row +
                       (pair ? 16u * (uint32_t)g + 32u * (uint32_t)s + 8u * e
                             : last_tile_bytes(NB, quad_feature(s + e - (4 * NB - 4), g), D)));
            }
        }
    }
  });
}

int main() {
  const int rows[] = {1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 49};
  for (int N : rows) {
    for (int D = 1; D <= 64; ++D) check<64>(N, D);
    for (int D = 65; D <= 128; ++D) check<128>(N, D);
  }
  std::printf("%ld bad reads\n", bad);
  return bad != 0;
}
"""


def test_every_read_of_x_stays_in_its_row(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "reads.cpp", tmp_path / "reads"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "geomjax_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
