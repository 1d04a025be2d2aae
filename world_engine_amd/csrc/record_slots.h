// A fixed set of records handed out to calls in flight (bindings.cpp).  Host code, no Python and no
// HIP in it.
#pragma once
#include <atomic>
#include <chrono>
#include <cstdint>
#include <thread>

namespace we {

class RecordSlots {
 public:
  static constexpr int kCount = 32;

  // A free record's index, or -1 when every one is out.
  int try_take() {
    uint32_t b = busy_.load(std::memory_order_relaxed);
    while (~b != 0u) {
      const int slot = __builtin_ctz(~b);
      if (busy_.compare_exchange_weak(b, b | (1u << slot), std::memory_order_acquire)) return slot;
    }
    return -1;
  }
  // The same, waiting for one where none is free.  Calls that hold a record need the interpreter's lock
  // before they can give it back, so the wait must not be made under it: `unlocked(f)` runs f without.
  template <typename Unlocked>
  int take(Unlocked&& unlocked) {
    int slot = try_take();
    if (slot < 0)
      unlocked([&] {
        while ((slot = try_take()) < 0) std::this_thread::sleep_for(std::chrono::microseconds(20));
      });
    return slot;
  }
  void give_back(int slot) { busy_.fetch_and(~(1u << slot), std::memory_order_release); }

 private:
  std::atomic<uint32_t> busy_{0};
};

}  // namespace we
