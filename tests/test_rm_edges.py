"""The rules at the edges of the row-major GEMM tiles (csrc/rm_edges.h), compiled on the host with
g++ and asked over small shapes. A slab of B is taken in 16-byte loads where it is whole and ends at
or before the rows that are checked; none of these loads may leave the memory that holds B: the
16-byte granules from its first element to the last row's last."""
import subprocess

from conftest import PKG

LOADS = r'''
#include "rm_edges.h"
#include <algorithm>
#include <cstdio>
template <int CH>
int sweep(int BK) {
  for (int base = 0; base < CH; ++base)  // elements past a 16-byte boundary
    for (int n = 1; n <= 9; ++n)
      for (long ldb = n; ldb <= n + 5; ++ldb)
        for (int K = 1; K <= 3 * BK + 5; ++K) {
          const int k16 = K - rm_checked_rows<CH>(n, ldb, base % CH == 0 && ldb % CH == 0);
          const long end = (K - 1) * ldb + n, granule = (base + end + CH - 1) / CH * CH - base;
          for (int kb = 0; kb + BK <= std::min(K, k16); kb += BK)
            for (int r = kb; r < kb + BK; ++r)
              for (int c = 0; c < n; c += CH)
                if (r * ldb + c + CH > granule) {
                  printf("CH %d BK %d base %d n %d ldb %ld K %d: row %d reads past B\n", CH, BK, base, n, ldb, K, r);
                  return 1;
                }
        }
  return 0;
}
int main() {
  if (sweep<4>(32) || sweep<4>(64) || sweep<2>(16) || sweep<2>(32)) return 1;
  printf("ok\n");
  return 0;
}
'''


def run(tmp_path, text):
    src, exe = tmp_path / "edges.cpp", tmp_path / "edges"
    src.write_text(text)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", str(PKG / "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_no_load_of_b_leaves_its_memory(tmp_path):
    run(tmp_path, LOADS)


GRIDS = r'''
#include "rm_edges.h"
#include <cstdio>
int main() {
  const int totals[] = {1, 7, 255, 256, 100000, 4194303, 4194304, 8388609, 16777216, 33554433, 2147483647};
  const int wanted[] = {0, 1, 5, 512, 4194304, 20000000, 2147483647};
  for (int threads = 256; threads <= 1024; threads *= 2)
    for (int total : totals)
      for (int want : wanted) {
        const int g = rm_grid(want, total, threads);
        const bool capped = want > 0 && want < total ? g < want : g < total;
        if (g < 1 || g > total || (want > 0 && g > want) || (long)g * threads >= 1L << 32 || (capped && g % 8) ||
            (capped && (long)(g + 8) * threads < 1L << 32)) {
          printf("total %d wanted %d threads %d: %d\n", total, want, threads, g);
          return 1;
        }
      }
  printf("ok\n");
  return 0;
}
'''


def test_launches_stay_below_two_to_the_32_threads(tmp_path):
    run(tmp_path, GRIDS)
