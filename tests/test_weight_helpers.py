"""What a projection's helper workgroups ask for (world_engine_amd/csrc/fetch_ahead.h): rows of their own XCD's tiles, none
behind the last feature, none twice, no more per step than a tile takes in on average, and an end to it on every XCD, with
a tile or without."""
import os
import shutil
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "world_engine_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "fetch_ahead.h"

int main() {
  long cases = 0, wrong = 0;
  const int widths[] = {32, 64, 128}, steps[] = {1, 2, 3, 4, 5, 10, 16, 64};
  for (int rows : widths) for (int n_tiles = 1; n_tiles <= 130; n_tiles += n_tiles < 20 ? 1 : 11)
    for (int helpers = 1; helpers <= 8; ++helpers) for (int xcd = 0; xcd < 8; ++xcd) for (int nc : steps) {
      const we::AheadOrder o(n_tiles, xcd, helpers, rows);
      std::vector<int> seen(n_tiles * rows / 4, 0);
      long turns = 0, asked = 0;
      for (int k = 0; k < helpers; ++k) for (int w = 0; w < 8; ++w)
        for (int c = 1; c < nc && turns < 1000000; c += o.every, ++turns)
          for (int q = k * 8 + w; q < o.quads; q += helpers * 8) {
            const int row = o.row(q);
            ++asked;
            if (row < 0 || row + 4 > n_tiles * rows || (row / rows) % 8 != xcd) { ++wrong; continue; }
            if (c == 1) ++seen[row / 4];
          }
      wrong += turns >= 1000000 || asked > (long)((nc - 2) / o.every + 1) * o.quads;
      wrong += (long)o.quads > (long)o.every * helpers * ((64 + rows) / 4);
      for (int t = 0; t < n_tiles; ++t) for (int i = 0; i < rows / 4; ++i)
        wrong += nc > 1 && seen[t * rows / 4 + i] != (t % 8 == xcd);
      ++cases;
    }
  for (int tiles = 0; tiles <= 40; ++tiles) for (int steps_ = 1; steps_ <= 64; ++steps_) for (int fl = 2; fl <= 5; ++fl) {
    const int h = we::helpers_of(tiles, 256, steps_, fl);
    wrong += (h != 0 && h != 8) || (h > 0 && tiles + h > 32);
  }
  printf("%ld %ld\n", cases, wrong);
  return 0;
}
"""


def test_helpers_ask_for_their_tiles_rows_and_come_to_an_end(tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    src, exe = tmp_path / "ahead.cpp", tmp_path / "ahead"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    cases, wrong = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.split())
    assert cases > 10000 and wrong == 0
