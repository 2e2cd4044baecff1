"""Where the threads of a partial stage tile stand (solar_amd/csrc/solar_tiles.hpp):
on the CPU, for every panel size the partial tiles take.  The stage reads the
LDS cells up to three columns and rows around a thread's point, so a point
outside the tile's rows reads past the LDS arrays (the block has more threads
than the tile has points)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "solar_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "solar_tiles.hpp"
// a point of thread t in a tile w wide: the surplus threads at a row of their own
struct Loose { int tx, ty; bool own; };
static Loose loose(int t, int w, int) { return {t % w, t / w, true}; }
template <typename F>
static int bad(F point) {
  constexpr int TI = 64, TJ = 8;  // the LDS tiles: TJ + 6 rows (v_xi: TJ) of TI + 6
  int wrong = 0;
  for (int nr : {1, 24})
    for (int n = 17; n <= 512; ++n) {
      if (n % 16 == 0) continue;
      const int w = solar::part_width(n, nr), nth = solar::part_threads(w, TJ);
      bool ok = w >= 1 && w <= TI && nth <= TI * TJ && nth % 64 == 0;
      std::vector<int> owners(w * TJ, 0);
      for (int t = 0; t < nth; ++t) {
        const auto p = point(t, w, TJ);
        const bool in = p.tx >= 0 && p.tx < w && p.ty >= 0 && p.ty < TJ;
        ok = ok && in;
        if (in && p.own) ++owners[p.ty * w + p.tx];
      }
      for (int o : owners) ok = ok && o == 1;
      wrong += !ok;
    }
  return wrong;
}
int main() { std::printf("%d %d\n", bad(solar::part_point), bad(loose)); }
"""


@pytest.fixture(scope="module")
def counts(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", CSRC, str(d / "p.cpp"), "-o", str(d / "p")], check=True)
    return [int(v) for v in subprocess.run([str(d / "p")], capture_output=True, text=True, check=True).stdout.split()]


def test_every_thread_stands_in_the_tile_and_every_point_has_one_owner(counts):
    assert counts[0] == 0


def test_the_check_sees_threads_past_the_rows(counts):
    assert counts[1] > 0
