// What the launchers of the LDS-staged kernels share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace nplm {

// Tiles above 64 KiB need the dynamic-LDS limit of their kernel raised: once per kernel and device
// (`done` is a static of the calling launcher, one per kernel instantiation; bit d = done on device d).
template <typename KernelT>
hipError_t allow_lds(std::atomic<uint64_t>& done, KernelT kernel, size_t shmem) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

}  // namespace nplm
