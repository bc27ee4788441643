// Host side of the 16-bit grouped GEMM launches.
#pragma once

#include "gemm_common.h"

namespace {

// compute units of the current device (0 if it cannot be read)
static int device_cu_count()
{
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// The few-row kernel's 16-row tiles: 64 columns and eight wavefronts each where 128 columns and four do not give every compute unit
// one (one token), 128 and four otherwise
static bool skinny_narrow(int m_tiles, int N, int cus) { return (long long)m_tiles * ((N + 127) / 128) < cus; }

template <auto KERN, int THREADS, int LDS_BYTES>
int launch_kernel(const GemmArgs& a, int grid, hipStream_t s)
{
    // The LDS limit is an attribute of the kernel on one device: set once per device (bit d of the
    // mask); setting it twice from racing threads is harmless.
    static std::atomic<unsigned long long> attr_done{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 63;   // 63: never cached
    if (dev == 63 || !(attr_done.load(std::memory_order_relaxed) >> dev & 1ull)) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(KERN),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
        if (err != hipSuccess) {
            amoe_set_error("grouped_gemm: cannot reserve %d bytes of LDS: %s", LDS_BYTES, hipGetErrorString(err));
            return AMOE_ERR_LAUNCH;
        }
        if (dev != 63) attr_done.fetch_or(1ull << dev, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL(KERN, dim3(grid), dim3(THREADS), LDS_BYTES, s, a);
    return amoe_check_launch("grouped_gemm_16bit");
}

}  // namespace
