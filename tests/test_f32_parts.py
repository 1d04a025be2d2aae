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


LAUNCHED = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include "attn_plan.h"

static int parts, groups;
namespace we {
hipError_t launch_attn_ring_f32(const AttnParams& p, int, int q_groups, int, hipStream_t) {
  parts = p.n_splits;
  groups = q_groups;
  return hipSuccess;
}
#define OTHER(name, ...) hipError_t name(const AttnParams&, __VA_ARGS__, hipStream_t) { return hipErrorUnknown; }
OTHER(launch_attn_ring_bf16_128, int) OTHER(launch_attn_ring_bf16_64, int) OTHER(launch_attn_ring_f16_128, int) OTHER(launch_attn_ring_f16_64, int)
OTHER(launch_attn_ring_short_bf16, int, int) OTHER(launch_attn_ring_short_f16, int, int) OTHER(launch_attn_ring_shared_bf16, int, int)
OTHER(launch_attn_ring_shared_f16, int, int) OTHER(launch_attn_combine, int, int)
}

int main() {
  long cases = 0, wrong = 0, less = 0;
  const int64_t st[3] = {1 << 20, 1 << 10, 128};
  uint8_t* at = reinterpret_cast<uint8_t*>(4096);   // (no memory is touched)
  int64_t* t_pos = reinterpret_cast<int64_t*>(at);
  for (int heads : {1, 2, 3, 8, 16, 40}) for (int T : {16, 33, 64, 256}) for (int slots : {2, 8, 16, 64}) for (int dh : {64, 128})
    for (int d : {1, 2}) for (int share : {0, 16, 8, 4, 2, 1}) for (int splits : {0, 1}) {
      we::F32Call want = {heads, T, slots / d, dh, 256};
      want.plan(INT64_MAX);
      const int64_t all = want.bytes(want.parts), given = share ? all / share : 0;
      want.plan(splits ? 0 : given);
      we::AttnParams p;
      we::host::AttnPlan pl;
      const int rc = we::host::prepare_attn(at, st, at, at, t_pos, at, st, given ? at : nullptr, (size_t)given, 1, heads, heads, T, dh,
                                            (int64_t)slots * T, d, 0.1f, splits, 0, WE_DTYPE_F32, 256, p, pl);
      parts = groups = 0;
      wrong += rc != WE_OK || we::host::launch_attn(p, pl, dh, WE_DTYPE_F32, nullptr) != WE_OK;
      wrong += parts != want.parts || groups != want.groups || (parts > 1 && want.bytes(parts) > given);
      if (share > 1 && parts > 1) ++less;
      ++cases;
    }
  printf("%ld %ld %ld\n", cases, wrong, less);
  return 0;
}
"""


def test_what_is_launched_is_what_was_planned(tmp_path):
    """Parts and groups of queries together, also with a workspace that holds fewer parts than the best plan has."""
    cxx, rocm = os.environ.get("CXX") or shutil.which("g++"), os.environ.get("ROCM_PATH", "/opt/rocm")
    src, exe = tmp_path / "launched.cpp", tmp_path / "launched"
    src.write_text(LAUNCHED)
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__=1", f"-I{CSRC}", f"-isystem{rocm}/include", str(src), "-o", str(exe)],
                   check=True)
    cases, wrong, less = map(int, subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.split())
    assert cases > 1000 and less > 50 and wrong == 0


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
