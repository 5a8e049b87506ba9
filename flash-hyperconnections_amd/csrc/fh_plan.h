// Launch arithmetic with no device in it.
#pragma once
#include <atomic>
#include <cstdint>

namespace fh {

// A positive property of every device, asked for once a device.  A query that fails
// (gives nothing positive) counts as 1 and is asked again.
class PerDevice {
 public:
  template <typename Query>
  int64_t get(int device, Query query) {
    const bool known = device >= 0 && device < kDevices;
    int value = known ? values_[device].load(std::memory_order_relaxed) : 0;
    if (value <= 0) {
      value = query();
      if (known && value > 0) values_[device].store(value, std::memory_order_relaxed);
    }
    return value > 0 ? value : 1;
  }

 private:
  static constexpr int kDevices = 64;
  std::atomic<int> values_[kDevices] = {};
};

}  // namespace fh
