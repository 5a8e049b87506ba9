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

// Bytes from the first token's operands of a stream mixing to those of token
// `first`: h, x and gy by their batch strides (elements of `es` bytes), the
// contiguous results [B, n, C], [B, n, n] and, in FP32, [B, n, n].
struct MixBytes {
  int64_t h, x, gy, rows, square, square_f32;
};
inline MixBytes mix_bytes(int64_t first, int64_t es, int64_t n, int64_t cols, int64_t hb, int64_t xb, int64_t gb) {
  return {first * hb * es, first * xb * es, first * gb * es, first * n * cols * es, first * n * n * es, first * n * n * 4};
}

// f(first, count) for consecutive slices of at most `most` of `batch` tokens, up to
// the first that does not return zero.
template <typename F>
auto in_slices(int64_t batch, int64_t most, F f) {
  for (int64_t first = 0;; first += most) {
    const int64_t left = batch - first;
    const auto status = f(first, left < most ? left : most);
    if (static_cast<int>(status) != 0 || left <= most) return status;
  }
}

}  // namespace fh
