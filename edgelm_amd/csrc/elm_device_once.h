// A set-up step that has to run once on each device (plain C++, no HIP: a kernel's raised dynamic-LDS limit holds for the
// device that was current when it was raised, and contexts of one process may be on several).
#pragma once
#include <atomic>
#include <cstdint>
#include <mutex>

namespace elmh {

class DeviceOnce {
 public:
  // True once step() has returned true on this device: it runs at the device's first call, and again at later calls for as
  // long as it returns false. Calls of several threads are safe; a device past the 64th has its step run on every call.
  template <class F>
  bool run(int device, F&& step) {
    if (device < 0 || device >= 64) return step();
    const uint64_t bit = uint64_t(1) << device;
    if (done_.load(std::memory_order_acquire) & bit) return true;
    std::lock_guard<std::mutex> lock(mu_);
    if (done_.load(std::memory_order_relaxed) & bit) return true;
    if (!step()) return false;
    done_.fetch_or(bit, std::memory_order_release);
    return true;
  }

 private:
  std::atomic<uint64_t> done_{0};
  std::mutex mu_;
};

}  // namespace elmh
