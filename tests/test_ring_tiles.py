"""What a split of the context asks for (world_engine_amd/csrc/ring_tiles.h): every key of its own once, and never a
row behind the last key there is, however short the context and however many its parts."""
import os
import shutil
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "world_engine_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "ring_tiles.h"

int main() {
  long cases = 0, wrong = 0;
  const int sizes[] = {64, 65, 72, 100, 127, 129, 143, 200, 225, 300, 374, 720};
  for (int T : sizes) for (int nvis = 1; nvis <= 17; nvis += nvis < 5 ? 1 : 4) for (int nsp = 1; nsp <= 24; ++nsp)
    for (unsigned g = 1; g <= 4; g *= 2) for (unsigned m = 0; m < g; ++m) {
      const int keys = nvis * T, nt = (keys + 63) / 64, last = keys - (nt - 1) * 64;
      std::vector<int> seen(nt, 0);
      for (int sp = 0; sp < nsp; ++sp) {
        const unsigned b = sp * nt / nsp, e = (sp + 1) * nt / nsp;
        if (e == b) continue;
        const we::SplitTiles s = {b, e, (int)e == nt && last < 64, g, m};
        int k = 0;
        for (int r = 0; r < (int)s.count() + 6; ++r) {      // the pipeline's requests run past the end of the split
          const unsigned t = s.at((unsigned)k);
          const int rows = r == 0 && s.shorted ? last : 64;
          if (t * 64 + rows > (unsigned)keys || (r < (int)s.count() && (t < b || t >= e))) ++wrong;
          if (r < (int)s.count()) ++seen[t];
          k = s.next(k);
        }
      }
      for (int n : seen) wrong += n != 1;
      ++cases;
    }
  printf("%ld %ld\n", cases, wrong);
  return 0;
}
"""


def test_every_tile_once_and_no_row_past_the_last_key(tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    cases, wrong = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.split())
    assert cases > 10000 and wrong == 0
