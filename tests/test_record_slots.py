"""Calls in flight beyond the number of records (world_engine_amd/csrc/record_slots.h): the ones that wait must not
keep the interpreter's lock, which the ones that hold a record need to give it back.  A host program plays the
binding with a mutex in the lock's place: more threads than records, each taking a record under the lock, waiting
without it and giving the record back under it."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "world_engine_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>
#include "record_slots.h"

int main(int argc, char** argv) {
  const int threads = atoi(argv[1]), calls = atoi(argv[2]);
  we::RecordSlots slots;
  std::mutex lock;
  std::atomic<int> holders[we::RecordSlots::kCount] = {};
  std::atomic<int> twice{0}, done{0};
  std::vector<std::thread> pool;
  for (int i = 0; i < threads; ++i)
    pool.emplace_back([&] {
      for (int c = 0; c < calls; ++c) {
        lock.lock();
        const int s = slots.take([&](auto&& wait) { lock.unlock(); wait(); lock.lock(); });
        if (s < 0 || s >= we::RecordSlots::kCount || holders[s]++ != 0) twice++;
        lock.unlock();                                                    // the verdict is waited for without the lock
        std::this_thread::sleep_for(std::chrono::milliseconds(2));
        lock.lock();
        holders[s]--;
        slots.give_back(s);
        done++;
        lock.unlock();
      }
    });
  for (auto& t : pool) t.join();
  printf("%d %d\n", done.load(), twice.load());
  return 0;
}
"""


@pytest.mark.parametrize("threads", [1, 32, 33, 100])
def test_more_calls_than_records_all_finish(tmp_path, threads):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe), str(threads), "5"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.split() == [str(threads * 5), "0"], out.stdout + out.stderr
