// Leave for a kernel to take more than 64 KB of dynamic LDS. The HIP attribute belongs to a function on one
// device, so a process that uses several devices has to set it on each; it is set once per device and
// function, by whichever thread comes first (setting it twice is harmless).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

namespace qmm4 {

class LdsAllowance {
 public:
  // Calls set() unless it has succeeded for device `dev` before.
  template <class Set>
  hipError_t once(int dev, Set&& set) {
    const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t{1} << dev : 0;
    if (done_.load(std::memory_order_acquire) & bit) return hipSuccess;
    const hipError_t e = set();
    if (e == hipSuccess) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }

  hipError_t allow(const void* f, size_t bytes) {
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    return once(dev, [&] { return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes); });
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace qmm4
