"""How an fp32 call is cut up (world_engine_amd/csrc/f32_parts.h): one round of workgroups where there are parts, partial rows
that the workspace holds, every part with keys, two groups of queries in one pass only where one would not fit the CUs."""
import os
import shutil
import subprocess

from world_engine_amd import _capi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "world_engine_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "f32_parts.h"

int main() {
  long cases = 0, wrong = 0;
  for (int cus : {64, 256, 304}) for (int heads : {1, 2, 3, 8, 16, 40, 100}) for (int T : {1, 15, 16, 33, 64, 256, 1000})
    for (int slots : {1, 2, 5, 16, 64, 256}) for (int dh : {64, 128}) for (long long most : {0ll, 100000ll, 4000000ll, 1ll << 60}) {
      we::F32Call c = {heads, T, slots, dh, cus};
      c.plan(most);
      wrong += c.parts < 1 || c.parts > 16 || c.groups < 1 || c.groups > 2;
      wrong += c.parts > 1 && (c.tiles(c.groups) * c.parts > cus || c.blocks() / c.parts < 8 || c.bytes(c.parts) > most);
      wrong += c.parts > 1 && !(c.cost(c.groups, c.parts) < c.cost(1, 1));
      wrong += c.parts == 1 && (c.groups == 2) != (c.tiles(1) > cus && c.blocks() >= c.halves_from());
      wrong += c.bytes(1) != 0;
      ++cases;
    }
  printf("%ld %ld\n", cases, wrong);
  return 0;
}
"""


def test_parts_and_groups(tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    src, exe = tmp_path / "parts.cpp", tmp_path / "parts"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    cases, wrong = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.split())
    assert cases > 1000 and wrong == 0


def test_workspace_of_an_fp32_call():
    lib = _capi.lib()
    bytes_of = lib.we_attn_f32_workspace_bytes
    assert bytes_of(1, 4, 4, 128, 128, 16 * 128, 1) % (4 * 128 * (128 * 4 + 8)) == 0 < bytes_of(1, 4, 4, 128, 128, 16 * 128, 1)
    assert bytes_of(1, 4, 4, 128, 128, 16 * 128, 16) == 0           # one slot's keys
    assert bytes_of(1, 8, 8, 64, 64, 4 * 64, 1) == 0                # a short context of narrow heads
    assert bytes_of(1, 24, 24, 1024, 128, 8 * 1024, 1) == 0         # more workgroups than CUs
    for bad in ((0, 4, 4, 128, 128, 2048, 1), (1, 4, 3, 128, 128, 2048, 1), (1, 4, 4, 128, 96, 2048, 1), (1, 4, 4, 128, 128, 2000, 1),
                (1, 4, 4, 128, 128, 2048, 3)):
        assert bytes_of(*bad) == 0, bad
