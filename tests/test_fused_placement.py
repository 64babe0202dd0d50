"""Which XCD's L2 the fused pass's launches bring the next launch's matrix
columns into (csrc/sevp_tiles.h): the columns must be those that the next
launch's product workgroups on that XCD read, whatever the heights of the two
blocks and the workgroups of the homogeneous march that come first.  The
header is built alone with g++, so this runs without a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "musoc_solver_amd", "csrc")

# One line per case: i2, periodic, row-tile groups, steps of this forward launch and the next one;
# wavefronts of homogeneous march in this backward launch and the next one, wavefronts a workgroup.
# Prints, for each direction, per XCD the columns brought near and the columns read.
HARNESS = r"""
#include <cstdio>
#include <set>
#include "sevp_tiles.h"
using namespace sevp;
typedef std::set<int> Cols[8];
static void show(const Cols &c) {
  for (int x = 0; x < 8; ++x) {
    for (int v : c[x]) std::printf("%d ", v);
    std::printf(";");
  }
  std::printf("\n");
}
int main() {
  int i2, per, nmb, steps, next, hom, homn, w, tile, mb;
  while (std::scanf("%d%d%d%d%d%d%d%d", &i2, &per, &nmb, &steps, &next, &hom, &homn, &w) == 8) {
    {
      Cols near, read;
      const int first = (int)placed_workgroups(fused_tiles_fwd(i2, steps), nmb);
      const int nt = fused_tiles_fwd(i2, next);
      for (int g = 0; g < placed_workgroups(nt, 1); ++g)
        if (warm_tile(g, nt, tile))
          for (int i = 0; i < 16; ++i)
            near[(first + g) % 8].insert(fused_fwd_matrix_column(fused_fwd_column(tile, next, i), i2, per));
      for (int g = 0; g < placed_workgroups(nt, nmb); ++g)
        if (tile_of(g, nt, nmb, tile, mb))
          for (int i = 0; i < 16; ++i)
            read[g % 8].insert(fused_fwd_matrix_column(fused_fwd_column(tile, next, i), i2, per));
      show(near);
      show(read);
    }
    {
      Cols near, read;
      const int nt = (i2 + 15) / 16, half = (int)placed_workgroups(nt, nmb);
      const int first = march_workgroups(hom, w) + 2 * half, prod = march_workgroups(homn, w);
      for (int g = 0; g < placed_workgroups(nt, 1); ++g)
        if (warm_tile(g, nt, tile))
          for (int i = 0; i < 16; ++i) near[(first + g) % 8].insert(16 * tile + i);
      for (int g = 0; g < half; ++g)
        if (tile_of(g, nt, nmb, tile, mb))
          for (int i = 0; i < 16; ++i) read[(prod + g) % 8].insert(16 * tile + i);
      show(near);
      show(read);
    }
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("placement")
    src, exe = d / "placement.cpp", d / "placement"
    src.write_text(HARNESS)
    subprocess.run([cxx, "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return str(exe)


def test_next_matrices_on_the_reading_xcd(harness):
    cases = [(i2, per, nmb, steps, nxt, hom, homn, w)
             for i2 in (16, 64, 200, 516, 1440) for per in (0, 1) for nmb in (1, 2, 4)
             for steps, nxt in ((1, 1), (1, 3), (3, 1), (0, 1), (1, 0), (2, 3))
             for hom, homn, w in ((0, 24, 16), (24, 24, 16), (24, 1500, 8), (5, 17, 16))]
    inp = "".join(" ".join(map(str, c)) + "\n" for c in cases)
    out = subprocess.run([harness], input=inp, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(out) == 4 * len(cases)
    for k, c in enumerate(cases):
        near_f, read_f, near_b, read_b = out[4 * k:4 * k + 4]
        assert any(read_f.split(";")) and near_f == read_f, c
        assert any(read_b.split(";")) and near_b == read_b, c
