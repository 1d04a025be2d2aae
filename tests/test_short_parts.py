"""How many context parts a short call takes (world_engine_amd/csrc/short_parts.h): at least one, never more than planned,
the planner's own count where nothing is gained, fewer for wider partial rows."""
import os
import shutil
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "world_engine_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "short_parts.h"

int main() {
  long cases = 0, wrong = 0;
  for (int cus : {8, 64, 256, 304}) for (int units = 1; units <= 200; units += units < 20 ? 1 : 23) for (int members : {1, 2, 3, 8})
    for (int tiles = 1; tiles <= 300; tiles += tiles < 10 ? 1 : 37) for (int planned = 1; planned <= 64; planned += planned < 8 ? 1 : 9)
      for (bool wide : {false, true}) {
        const int dh = wide ? 128 : 64;
        we::ShortCall c = {units, members, tiles, units * 128, 2 * dh + 16, wide, cus};
        const int half = c.parts(planned);
        c.row_bytes = 4 * dh + 16;
        const int full = c.parts(planned);
        wrong += half < 1 || half > planned || full < 1 || full > half;
        wrong += planned == 1 && half != 1;
        wrong += full != planned && !(c.cost(full) < c.cost(planned));
        ++cases;
      }
  // 16 heads of 128, 256 tokens, 16 slots keep their six parts; 13 units of 128 tokens and six slots run in one pass
  wrong += we::ShortCall{16, 2, 64, 4096, 272, true, 256}.parts(6) != 6;
  wrong += we::ShortCall{13, 2, 12, 26 * 128, 528, true, 256}.parts(6) != 1;
  printf("%ld %ld\n", cases, wrong);
  return 0;
}
"""


def test_parts_of_short_calls(tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    src, exe = tmp_path / "parts.cpp", tmp_path / "parts"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    cases, wrong = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.split())
    assert cases > 10000 and wrong == 0
