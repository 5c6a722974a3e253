// A setting that each device needs once (a kernel's LDS limit), made on the
// first use of every device and from any thread.
#pragma once
#include <atomic>
#include <cstdint>

namespace sma_abi {

class OncePerDevice {
  std::atomic<uint64_t> set_{0};   // bit d: made on device d

 public:
  // Calls make() unless it has succeeded (returned 0) for `dev`; returns its
  // result.  make() may run more than once: first uses by several threads at
  // once, devices beyond the 64th.
  template <class Make>
  int operator()(int dev, Make make) {
    const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t(1) << dev : 0;
    if (set_.load(std::memory_order_acquire) & bit) return 0;
    const int rc = make();
    if (rc == 0) set_.fetch_or(bit, std::memory_order_release);
    return rc;
  }
};

}  // namespace sma_abi
