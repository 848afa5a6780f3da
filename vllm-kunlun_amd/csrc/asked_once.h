// A host value that is asked for once per process (no GPU code).
#pragma once
#include <atomic>

namespace kmoe {

// Whichever call needs the value first asks for it; calls of several threads may do so at the same time, and each of them then
// stores the same answer.
class AskedOnce {
 public:
  // ask(): the value, positive; anything else is not kept, and the next call asks again
  template <class Ask>
  int get(Ask&& ask) {
    int value = value_.load(std::memory_order_relaxed);
    if (value <= 0) {
      value = ask();
      if (value > 0) value_.store(value, std::memory_order_relaxed);
    }
    return value;
  }

 private:
  std::atomic<int> value_{0};
};

}  // namespace kmoe
