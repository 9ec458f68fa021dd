// Dynamic LDS above 64 KiB: a kernel has to be opted in for it, on each device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

namespace mcrg {

// One kernel's level on each device.  Chains, batches and servers may launch from
// different threads: a level only ever rises, under a lock, so a launch never
// finds it lowered by another.
class LdsOptIn {
  public:
    // For a launch of `kernel` with `bytes` of dynamic LDS on the current device.
    hipError_t need(const void *kernel, uint32_t bytes)
    {
        if (bytes <= kFree) return hipSuccess;
        int device = 0;
        hipError_t e = hipGetDevice(&device);
        if (e != hipSuccess) return e;
        std::lock_guard<std::mutex> lk(mu_);
        const bool known = device >= 0 && device < kDevices;
        if (known && bytes <= level_[device]) return hipSuccess;
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e == hipSuccess && known) level_[device] = bytes;
        return e;
    }

  private:
    static constexpr uint32_t kFree = 65536u;
    static constexpr int kDevices = 64;
    std::mutex mu_;
    uint32_t level_[kDevices] = {};
};

}  // namespace mcrg
