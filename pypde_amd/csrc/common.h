// Shared helpers for the pypde_amd HIP library (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdio>
#include <cstdarg>
#include <mutex>
#include <string>

namespace pypde {

// Thread-local last-error message returned by pypde_last_error().
void set_error(const char* fmt, ...);
const char* last_error();

enum Status : int {
    OK = 0,
    ERR_ARG = -1,     // invalid argument (shape, pointer, size)
    ERR_HIP = -2,     // HIP runtime error
    ERR_UNSUP = -3,   // unsupported configuration
};

inline int check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return ERR_HIP;
    }
    return OK;
}

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

constexpr int kWave = 64;

// Orders LDS traffic within one wavefront (other waves are not synchronised).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroups are dispatched to the device's 8 XCDs in turn (workgroup i to
// XCD i mod 8), and each XCD has its own L2.  Renumbering them so that XCD x
// runs a contiguous range of work items keeps the cache lines that
// neighbouring items share (GEMM operand panels, the 128-byte lines that
// neighbouring columns of a row-major array share) in one L2 instead of
// fetching them into all eight.  The map is a bijection on [0, total):
// results do not change, only where the work runs.
constexpr int kXcd = 8;
__device__ __forceinline__ int xcd_remap(int pid, int total)
{
    const int q = total / kXcd, r = total - q * kXcd;
    const int x = pid % kXcd, local = pid / kXcd;
    return x * q + (x < r ? x : r) + local;
}

// Bytes of the device tables of the multi launches (one per translation unit).
long long gemm_multi_bytes();
long long recurrence_multi_bytes();
long long products_multi_bytes();

}  // namespace pypde

#define PYPDE_REQUIRE(cond, ...)                 \
    do {                                         \
        if (!(cond)) {                           \
            ::pypde::set_error(__VA_ARGS__);     \
            return ::pypde::ERR_ARG;             \
        }                                        \
    } while (0)

#define PYPDE_HIP(call)                                                        \
    do {                                                                       \
        hipError_t _e = (call);                                                \
        if (_e != hipSuccess) {                                                \
            ::pypde::set_error("%s: %s", #call, hipGetErrorString(_e));        \
            return ::pypde::ERR_HIP;                                           \
        }                                                                      \
    } while (0)

namespace pypde {

// Asks for `bytes` of dynamic LDS for a kernel, whose static LDS counts towards the
// default limit too: once per kernel, device and larger size, before its launch.
// The limit is only ever raised.
template <auto Kernel>
int allow_lds(size_t bytes)
{
    constexpr int kDevices = 64;
    static std::atomic<size_t> granted[kDevices];
    static std::mutex raising;
    int dev = 0;
    PYPDE_HIP(hipGetDevice(&dev));
    PYPDE_REQUIRE(dev >= 0 && dev < kDevices, "device %d not in 0..%d", dev, kDevices - 1);
    if (granted[dev].load(std::memory_order_acquire) >= bytes) return OK;
    std::lock_guard<std::mutex> lock(raising);
    if (granted[dev].load(std::memory_order_relaxed) >= bytes) return OK;
    PYPDE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    granted[dev].store(bytes, std::memory_order_release);
    return OK;
}

}  // namespace pypde
