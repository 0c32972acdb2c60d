"""The choice of a kernel for a device product (tiled-mm_amd/csrc/tmm_ksplit.h) against the limit of a launch: a grid holds
fewer than 2^32 threads, 256 for each tile."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include "tmm_ksplit.h"
#include <cmath>
#include <cstdio>
using namespace tmm;
int main() {
  const long edges[] = {1, 16, 17, 33, 48, 1000, 65537, 131072, 140001, 1L << 24, 1L << 28, (1L << 28) + 5, 1L << 29, 1L << 30, (1L << 31) - 1};
  int bad = 0, taken = 0;
  for (int t = 0; t < 4; ++t)
    for (long m : edges)
      for (long n : edges) {
        if ((double)m * n > 7e10) continue;  // 280 GB of the smallest type
        for (long k : {1L, 64L, 128L, 160L, 500L, 4000L}) {
          const KsType type = (KsType)t;
          long tiles;
          if (short_inner(type, m, n, k, 256)) {
            tiles = ks_tiles(kKsShapes[kShortShape], m, n);
          } else {
            double us = 0;
            const int shape = ks_shape(type, m, n, k, 256, &us);
            if (std::isinf(us)) continue;  // not taken
            tiles = ks_tiles(kKsShapes[shape], m, n);
          }
          ++taken;
          if (tiles * 256 >= 1L << 32 && ++bad < 10) std::printf("type %d %ld x %ld x %ld: %ld tiles\n", t, m, n, k, tiles);
        }
      }
  std::printf("%d of %d\n", bad, taken);
  return bad != 0 || taken < 1000;
}
"""


def test_chosen_tiles_fit_a_grid(tmp_path):
    src = tmp_path / "limits.cpp"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "tiled-mm_amd", "csrc"),
                    "-I" + rocm + "/include", str(src), "-o", str(tmp_path / "limits")], check=True)
    run = subprocess.run([str(tmp_path / "limits")], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
