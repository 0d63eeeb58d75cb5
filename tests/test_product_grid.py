"""Grid sizes of the solvers' products (libmesh_amd/csrc/lmh_grids.h), compiled for
the host: the partial sums of every grid fit the buffer, whatever the number of
CUs and the compiled-in workgroups per CU, and the grids of a 256-CU GPU are the
measured ones."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "libmesh_amd", "csrc")
SOURCE = r"""
#include <cstdio>
#include "lmh_grids.h"
int main() {
  using lmh::product_grid;
  int bad = 0;
  for (int cus : {1, 8, 64, 255, 256, 304, 341, 342, 512, 1024})
    for (int per_cu : {1, 4, 16, 32, 64, 128})
      for (int resident : {0, 5, 10})
        for (int n_part : {256, 4096, 16384})
          for (int64_t blocks : {1, 7, 8, 9, 1000, 2561, 10241, 24576, 140203, 1 << 30}) {
            const int64_t g = product_grid(cus, per_cu, resident, n_part, blocks);
            if (g < 1 || 3 * g > 2 * (int64_t)n_part || g > (int64_t)cus * per_cu || g > (blocks + 7) / 8 * 8) {
              ++bad;
              std::printf("cus %d per_cu %d resident %d n_part %d blocks %lld: %lld\n", cus, per_cu, resident, n_part,
                          (long long)blocks, (long long)g);
            }
          }
  // 256 CUs: 64^3 Q2 (140,203 blocks), 20^3 (4,050), 3 blocks, int32 columns (full grid)
  if (product_grid(256, 32, 10, 16384, 140203) != 8192 || product_grid(256, 32, 10, 16384, 4050) != 2032 ||
      product_grid(256, 32, 10, 16384, 3) != 8 || product_grid(256, 16, 5, 16384, 70000) != 4096)
    ++bad, std::printf("256-CU grids differ\n");
  // without rounds: a workgroup per block
  if (product_grid(256, 16, 0, 16384, 4000) != 4000) ++bad, std::printf("rounds where none are asked for\\n");
  return bad != 0;
}
"""


def test_partials_fit(tmp_path):
    src, exe = tmp_path / "grids.cpp", tmp_path / "grids"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
