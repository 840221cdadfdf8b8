// sa_per_device.hpp -- settings of a kernel that hold for one device (its limit of dynamic LDS).
#pragma once

#include <atomic>
#include <cstdint>

namespace sa {

// Acts once on each device, from any thread; an act that failed is tried again.
class per_device_once {
  std::atomic<uint64_t> done_{0};  // a bit per device; devices beyond 63 act every time

 public:
  // 0, or the act's error
  template <class Act>
  int operator()(int device, Act act) {
    const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
    if (done_.load(std::memory_order_acquire) & bit) return 0;
    const int e = (int)act();
    if (!e) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }
};

}  // namespace sa
