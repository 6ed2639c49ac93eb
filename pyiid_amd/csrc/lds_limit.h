// Dynamic LDS beyond 64 KB has to be asked for, for every kernel on every device.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace pyiid {

// Which devices a launcher's kernels have been allowed their LDS on; one static object
// per launcher.
class LdsLimit {
 public:
  // The kernels may use up to `bytes` on the current device from now on.
  hipError_t allow(std::initializer_list<const void*> kernels, size_t bytes) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const uint64_t bit = device < 64 ? uint64_t(1) << device : 0;  // others: every time
    if (done_.load(std::memory_order_acquire) & bit) return hipSuccess;
    for (const void* k : kernels) {
      e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
      if (e != hipSuccess) return e;
    }
    done_.fetch_or(bit, std::memory_order_release);
    return hipSuccess;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace pyiid
