// lds_optin.h — the opt-in that kernels with more than 64 KiB of dynamic LDS need.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>

namespace rk {

// Lets `kern` be launched with `bytes` of dynamic LDS on the current device, once per device (bit d of
// `opted`, one mask a kernel; any thread may launch, so the mask is atomic).
inline hipError_t lds_opt_in(const void *kern, int bytes, std::atomic<uint64_t> &opted)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipGetLastError();
    const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t)1 << dev : 0;
    if (!bit || !(opted.load(std::memory_order_acquire) & bit)) {
        if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return hipGetLastError();
        opted.fetch_or(bit, std::memory_order_release);
    }
    return hipSuccess;
}

}  // namespace rk
