"""Address arithmetic of the kernels, checked on the host.

The functions of ``csrc/addressing.h`` that the kernels call are compiled with
the host compiler and walked over every lane and slot, for every fine-grid
length an axis can have, up to grids of 2^30 cells.
"""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mri-nufft_amd", "csrc")


def run_check(tmp_path, body):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text('#include <algorithm>\n#include <cstdio>\n#include <cstdlib>\n'
                   '#include "addressing.h"\nusing namespace hn;\n' + body)
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


STRIDED = r"""
int main() {
  long checked = 0;
  for (int n = 4; n <= 2730; n += 2) {
    int m = n;
    for (int p : {2, 3, 5}) while (m % p == 0) m /= p;
    if (m != 1) continue;
    const int64_t most = std::min<int64_t>((((int64_t)1 << 30) - 1) / n, 2730 * 2730);
    const int64_t lim32 = ((int64_t)1 << 29) / n;  // 4 GiB lines
    for (int64_t ls : {(int64_t)1, (int64_t)n, most / 2, lim32 - 1, lim32, lim32 + 1, most}) {
      if (ls < 1 || ls > most) continue;
      for (int64_t nx : {(int64_t)1, std::min<int64_t>(ls, 37), std::min<int64_t>(ls, 2730)}) {
        {
          // lines past 32 bits: all of the axis's lines per workgroup, more than
          // 4 elements per thread (the only forms with 64-bit offsets)
          const int L = lines_per_wg(n, 8192), NT = n * L > 4096 ? 512 : 256;
          if (!strided_fits_32(n, ls, nx) && (lines_of(L, ls) != L || n * L <= 4 * NT)) {
            printf("64-bit lines: n %d ls %ld\n", n, (long)ls);
            return 1;
          }
        }
        // an axis has at least `ls` lines: the pass takes L or, with few of them, a quarter
        for (int L : {lines_per_wg(n, 8192), lines_of(lines_per_wg(n, 8192), ls)})
          for (int NT : {256, 512}) {
            const int E = NT / L, PW = 64 / L;
            for (int M : {0, 1, n / 4, n / 3, n / 2 - 1, n / 2, 4 * n / 5, n - 1, n})
              for (int i = 0; i * E < n; ++i)
                for (int t = 0; t < NT; t += 1 + (L > 2 && t % L == 0) * (L - 2)) {
                  const int l = t % L, e0 = t / L, w0 = t / 64 * PW + i * E;
                  const int e = e0 + i * E, hin = M / 2, lim = M ? M : n;
                  const int lc = (int)std::min<int64_t>(l, nx - 1);
                  const uint32_t thread = strided_thread_offset(e0, ls, lc);
                  // the stores: a uniform base per slot plus the thread's own offset
                  if (e < n && thread != (uint64_t)(e0 * ls + lc) * 8) {
                    printf("thread offset: n %d ls %ld L %d e0 %d\n", n, (long)ls, L, e0);
                    return 1;
                  }
                  if (w0 >= lim || !strided_fits_32(n, ls, nx)) continue;
                  // columns of the first and of the last workgroup of a row of nx
                  for (int cols : {(int)std::min<int64_t>(L, nx), (int)((nx - 1) % L + 1)}) {
                    const int c = std::min(l, cols - 1);
                    const int64_t off = strided_cell_offset(
                        strided_thread_offset(e0, ls, c), strided_slot_offset(i, E, hin, ls), e,
                        hin, (uint32_t)(n * ls * 8));
                    const int64_t pos = e - hin + (e < hin ? n : 0), end = ((n - 1) * ls + cols) * 8;
                    const int64_t bytes = strided_line_bytes(n, ls, cols);
                    ++checked;
                    // a store of the cell at pos by its own offset
                    if (e < lim && strided_thread_offset((int)pos, ls, c) != (pos * ls + c) * 8) {
                      printf("store: n %d M %d ls %ld e %d\n", n, M, (long)ls, e);
                      return 1;
                    }
                    // a position's load reads its cell; lanes past the last one
                    // load, if anything, a cell between the lines' ends
                    if (bytes != end ||
                        (e < lim ? off != (pos * ls + c) * 8 || off + 8 > bytes
                                 : off < bytes && (off < 0 || off % 8 || off + 8 > end))) {
                      printf("load: n %d M %d ls %ld nx %ld L %d NT %d e %d: %ld\n", n, M, (long)ls,
                             (long)nx, L, NT, e, (long)off);
                      return 1;
                    }
                  }
                }
          }
      }
    }
  }
  printf("%ld\n", checked);
  return checked > 1000000 ? 0 : 1;
}
"""


def test_strided_pass(tmp_path):
    run_check(tmp_path, STRIDED)


# the row table of every region that the kernel accepts: behind the region and
# behind the weights, inside the kernel's LDS
PAIRS = r"""
int main() {
  for (int rows = 1; rows <= kStreamRows; ++rows)
    for (int cells = 128; cells <= kPairCells; cells += 128) {
      const int t = pair_row_table(cells);
      if (t < cells || t < kPairWeightCells || t + rows > kPairCells + kStreamRows) {
        printf("region of %d cells, %d rows: table at %d\n", cells, rows, t);
        return 1;
      }
    }
  // the weights end where the last point's do
  return kPairWeightCells * 2 == kPairNT / 64 * 8 * kPairTrips * kPairWRow ? 0 : 1;
}
"""


def test_interp_pairs_lds(tmp_path):
    run_check(tmp_path, PAIRS)
