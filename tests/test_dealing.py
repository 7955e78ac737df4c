"""How the line solvers deal line groups to workgroups (csrc/dealing.hpp),
compiled for the host: every group, outer index and part is taken once, and
the two eight-line halves of a 128-byte cache line go to the same one of the
eight XCDs (workgroup id mod 8), in round-robin order and in runs, with and
without interleaved parts."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "emix3d_amd", "csrc")

PROGRAM = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include "dealing.hpp"
#include <cstdio>
#include <cstdlib>
#include <vector>

template <int LG, bool INTERLEAVED>
void table(int run, int gx, int gy, int gz) {
  std::vector<int> xcd(gx * gy * gz, -1);
  for (int id = 0; id < gx * gy * gz; id++) {
    int x = id % gx, y = id / gx % gy, z = id / (gx * gy);
    emx::deal_lines<LG, INTERLEAVED>(run, gx, gy, gz, x, y, z);
    int& t = xcd.at(x + gx * (y + gy * z));
    if (t >= 0) { std::puts("taken twice"); std::exit(1); }
    t = id % 8;
  }
  int pairs = 0, same = 0;
  for (int row = 0; row < gy * gz; row++)
    for (int x = 0; x + 1 < gx; x += 2) {
      pairs++;
      same += xcd[x + gx * row] == xcd[x + 1 + gx * row];
    }
  std::printf("%d %d\n", pairs, same);
}

int main(int argc, char** argv) {
  const int lg = std::atoi(argv[1]), il = std::atoi(argv[2]), run = std::atoi(argv[3]);
  const int gx = std::atoi(argv[4]), gy = std::atoi(argv[5]), gz = std::atoi(argv[6]);
  if (lg == 8) (il ? table<8, true> : table<8, false>)(run, gx, gy, gz);
  else (il ? table<16, true> : table<16, false>)(run, gx, gy, gz);
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("dealing")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t")],
                   check=True)

    def run(*args):
        r = subprocess.run([str(d / "t"), *map(str, args)], check=True, capture_output=True, text=True)
        return tuple(map(int, r.stdout.split()))
    return run


@pytest.mark.parametrize("gx,gy,gz", [(64, 64, 1), (64, 33, 2), (32, 41, 2), (16, 300, 1), (33, 40, 2),
                                      (13, 97, 4), (5, 7, 1), (1, 1, 1), (17, 64, 2), (6, 200, 1)])
@pytest.mark.parametrize("interleaved", [0, 1])
@pytest.mark.parametrize("run", [0, 1])
@pytest.mark.parametrize("lg", [8, 16])
def test_line_groups(deal, lg, run, interleaved, gx, gy, gz):
    pairs, same = deal(lg, interleaved, run, gx, gy, gz)
    if lg == 8 and run == 0:
        # all but those of a row's last, incomplete set of 16 groups
        assert same >= gx // 16 * 8 * gy * gz
    if run and gx % 2 == 0:
        # all but those at an XCD's end of a run, and the grid's last 128
        # workgroups
        assert same >= 0.75 * pairs - 64
