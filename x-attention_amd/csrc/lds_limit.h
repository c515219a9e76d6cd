// Host helper of the kernels that use more than 64 KiB of dynamic LDS.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace xattn {

// Raises a kernel's dynamic LDS limit to the CU's 160 KiB, once per device: the call is host work that every launch
// would otherwise repeat.
class LdsLimit {
 public:
  hipError_t raise(const void* kernel) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done_.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace xattn
