// Host side of a kernel launch.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>

namespace itk {

// Whether `Kernel` may be launched with `bytes` of dynamic LDS on the current device.  More than 64 KB has to be asked for, once
// per kernel and device: the runtime keeps the answer with the device's copy of the kernel, so one device's does not do for
// another.  Any thread may come first; a refusal is not kept.  `bytes` is the most that the kernel is launched with.  (The kernel
// is the template's argument: instances of one kernel template have one type, and would share what a type keeps.)
template <auto Kernel>
bool lds_allowed(size_t bytes) {
    if (bytes <= 64 * 1024) return true;
    static std::atomic<uint64_t> asked{0};      // a bit a device (those past 63 are asked each time)
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) {
        const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;
        if (asked.load(std::memory_order_acquire) & bit) return true;
        if (hipFuncSetAttribute((const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess) {
            asked.fetch_or(bit, std::memory_order_release);
            return true;
        }
    }
    (void)hipGetLastError();
    return false;
}

// a kernel as a value whose type says which one it is, for lambdas that launch one of several
template <auto Kernel>
struct KernelIs {
    static constexpr auto value = Kernel;
};

}  // namespace itk
