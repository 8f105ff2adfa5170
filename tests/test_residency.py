"""The rules that keep lattices in the last-level cache (csrc/residency.h) lie
between the measured sides: dense solves by their own lattices, an AMR root by
all that a macro-step goes through."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "residency.h"
static double refined(int q, double cells, int tile, double tiles) {
  return 1e-6 * (cells + tiles * tile) * (2 * q + 4) * 4;
}
int main() {
  using namespace lbm;
  const int t3 = 20 * 20 * 20, t2 = 20 * 20, n96 = 96 * 96 * 96, n80 = 80 * 80 * 80, n2 = 1024 * 1024;
  printf("%d%d%d%d%d %d%d%d%d%d%d\n",
         cache_resident(60, 200, 19, false), cache_resident(270, 200, 19, true), cache_resident(350, 200, 19, false),
         cache_resident(10, 256, 19, false), cache_resident(60, 256, 27, true),
         cache_resident_refined(refined(27, n96, t3, 17)), cache_resident_refined(refined(27, n96, t3, 69)),
         cache_resident_refined(refined(27, n80, t3, 60)), cache_resident_refined(refined(27, n80, t3, 100)),
         cache_resident_refined(refined(9, n2, t2, 4096)), cache_resident_refined(refined(9, n2, t2, 6553)));
}
"""


def test_rules_lie_between_the_measured_sides(tmp_path):
    src = tmp_path / "r.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "r")
    subprocess.check_call(["g++", "-std=c++17", "-I", os.path.join(ROOT, "getting-air_amd", "csrc"), str(src), "-o", exe])
    # measured faster in the cache (1) or streamed (0)
    assert subprocess.check_output([exe], text=True).split() == ["11000", "101010"]
