"""Which tile of which system a block of the 3D tile sweep works on (sa_tile_place.hpp), against
plain division: every tile grid of sides 8..256 and every system's first and last tile up to the
systems that one launch is given.  Host code only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <set>
#include <utility>
#include "sa_tile_place.hpp"
int main() {
  std::set<std::pair<int, int>> grids;
  for (int L = 8; L <= 256; ++L)
    for (int tx : {4, 8, 16, 32})
      for (int ty : {4, 8, 16, 32})
        if (tx <= L && ty <= L) grids.insert({(L + tx - 1) / tx, (L + ty - 1) / ty});
  grids.insert({1, 1});  // held whole
  long checked = 0, wrong = 0;
  for (auto g : grids) {
    const uint32_t ntx = g.first, per = ntx * g.second, rp = sa::tile_recip(per);
    const int rx = sa::small_recip((int)ntx);
    for (int threads : {64, 256, 1024}) {
      const int64_t n = sa::systems_per_launch(per, threads);
      if (n < 1 || (n * per + 7) / 8 * 8 * threads >= (int64_t)1 << 32) ++wrong;
    }
    const int64_t most = sa::systems_per_launch(per, 256);
    for (int64_t sys = 0; sys < most; ++sys)
      for (uint32_t r : {0u, per - 1}) {
        const uint32_t b = (uint32_t)sys * per + r;
        const sa::tile_place p = sa::place_tile(b, per, rp, ntx, rx);
        ++checked;
        if (p.sys != sys || p.by != r / ntx || p.bx != r % ntx) {
          if (wrong++ < 5) std::printf("ntx %u per %u tile %u: system %u (%u, %u)\n", ntx, per, b, p.sys, p.bx, p.by);
        }
      }
    for (uint32_t r = 0; r < per; ++r) {
      const sa::tile_place p = sa::place_tile(r, per, rp, ntx, rx);
      if (p.sys != 0 || p.by != r / ntx || p.bx != r % ntx) ++wrong;
    }
  }
  std::printf("%zu grids, %ld tiles, %ld wrong\n", grids.size(), checked, wrong);
  return wrong ? 1 : 0;
}
"""


def test_every_block_finds_its_tile(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src = tmp_path / "place.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "place"
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-I", os.path.join(ROOT, "simulated_annealing_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
