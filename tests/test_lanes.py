"""The kernels' index arithmetic (mercury_amd/csrc/lanes.hpp), compiled for
the host: rows that end at or near position 2^32 are walked once and left, the
positions of every lane together are the range; searches in lockstep read
inside the array, also for a list that is empty at its end."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "lanes.hpp"
// walk b e: the positions of the 16 lanes, four at a time, as the sum of
// their distances from b and their number; 1 is returned past 2^16 steps.
int walks(int argc, char **argv) {
  for (int i = 2; i + 1 < argc; i += 2) {
    const uint32_t b = std::strtoul(argv[i], nullptr, 10);
    const uint32_t e = std::strtoul(argv[i + 1], nullptr, 10);
    unsigned long long sum = 0, count = 0, out = 0, steps = 0;
    for (uint32_t lane = 0; lane < 16; ++lane)
      mgpm::lane_walk<16, 4>(
          b, e, lane, [&](const uint32_t(&at)[4], const bool(&ok)[4]) {
            if (++steps > 65536) std::exit(1);
            for (int u = 0; u < 4; ++u) {
              out += at[u] < b || at[u] >= e;
              if (ok[u]) {
                sum += at[u] - b;
                ++count;
              }
            }
          });
    std::printf("%llu %llu %llu\n", sum, count, out);
  }
  return 0;
}
// search steps (lo end ok)...: what a search of each list reads in the
// array while the longest of them all halves `steps` times, as
// the lowest and the highest position.
int searches(int argc, char **argv) {
  const int steps = std::atoi(argv[2]);
  for (int i = 3; i + 2 < argc; i += 3) {
    mgpm::Window w = mgpm::search_window(
        std::strtoul(argv[i], nullptr, 10), std::strtoul(argv[i + 1], nullptr, 10),
        std::atoi(argv[i + 2]) != 0);
    uint32_t low = w.lo, high = w.lo;
    for (int k = 0; k < steps; ++k) {  // every entry is low enough
      const uint32_t at = w.lo + (w.len >> 1);
      if (at > high) high = at;
      w.lo = at;
      w.len -= w.len >> 1;
    }
    std::printf("%u %u\n", low, high);
  }
  return 0;
}
int main(int argc, char **argv) {
  return argv[1][0] == 'w' ? walks(argc, argv) : searches(argc, argv);
}
"""


@pytest.fixture(scope="module")
def lanes_bin(tmp_path_factory):
    d = tmp_path_factory.mktemp("lanes")
    src = d / "drv.cc"
    src.write_text(DRIVER)
    exe = d / "drv"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas",
                    f"-I{ROOT / 'mercury_amd' / 'csrc'}", str(src), "-o",
                    str(exe)], check=True)
    return exe


def test_rows_up_to_the_last_position(lanes_bin):
    top = 2**32 - 2  # entries come in pairs, fewer than 2^32 of them
    ranges = [(top - k, top) for k in (0, 1, 13, 14, 15, 16, 63, 64, 65, 1000)]
    ranges += [(top - 40, top - 40), (top - 40, top - 17), (0, 0), (0, 1),
               (7, 71), (100, 100 + 64 * 37 + 5)]
    args = [str(x) for r in ranges for x in r]
    run = subprocess.run([str(lanes_bin), "walk", *args], capture_output=True,
                         text=True)
    assert run.returncode == 0
    for (b, e), line in zip(ranges, run.stdout.splitlines(), strict=True):
        n = e - b
        assert [int(x) for x in line.split()] == [n * (n - 1) // 2, n, 0]


def test_searches_stay_inside_the_array(lanes_bin):
    m = 4096
    lists = [(m, m, 1), (m, m, 0), (17, 17, 1), (m - 1, m, 1), (m - 1, m, 0),
             (0, m, 1), (5, 69, 1), (m - 64, m, 1), (0, 1, 1)]
    out = subprocess.run(
        [str(lanes_bin), "search", "13", *(str(x) for q in lists for x in q)],
        capture_output=True, text=True, check=True).stdout
    for (lo, end, ok), line in zip(lists, out.splitlines(), strict=True):
        low, high = (int(x) for x in line.split())
        assert high < m
        if ok and end > lo:
            assert (low, high) == (lo, end - 1)
