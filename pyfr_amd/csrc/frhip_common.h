// Shared helpers for the frhip library (internal header).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>
#include <type_traits>

#include "../../include/frhip.h"

namespace frhip {

void set_error(const std::string &msg);

// Return a nonzero status with a message if a HIP call failed.
#define FR_HIP(call)                                                        \
    do {                                                                    \
        hipError_t _e = (call);                                             \
        if (_e != hipSuccess) {                                             \
            frhip::set_error(std::string(#call) + ": " +                    \
                             hipGetErrorString(_e));                        \
            return 1;                                                       \
        }                                                                   \
    } while (0)

#define FR_CHECK(cond, msg)                                                 \
    do {                                                                    \
        if (!(cond)) {                                                      \
            frhip::set_error(msg);                                          \
            return 2;                                                       \
        }                                                                   \
    } while (0)

// Launch-error check after a kernel launch.
#define FR_LAUNCHED()                                                       \
    do {                                                                    \
        hipError_t _e = hipGetLastError();                                  \
        if (_e != hipSuccess) {                                             \
            frhip::set_error(std::string("kernel launch: ") +               \
                             hipGetErrorString(_e));                        \
            return 3;                                                       \
        }                                                                   \
    } while (0)

// Catch-all so that no C++ exception crosses the ABI.
#define FR_API_BEGIN try {
#define FR_API_END                                                          \
    } catch (const std::exception &ex) {                                    \
        frhip::set_error(std::string("exception: ") + ex.what());           \
        return 9;                                                           \
    } catch (...) {                                                         \
        frhip::set_error("unknown exception");                              \
        return 9;                                                           \
    }

constexpr int SOA = 64;  // SoA width = gfx950 wavefront size

// Index of (element e, variable v) within one row of an AoSoA array.
__host__ __device__ inline long soa_ix(long e, int v, int nvar)
{
    return ((e >> 6) * nvar + v) * SOA + (e & 63);
}

// Workgroup index with each XCD given a contiguous range: workgroups are
// dispatched to the 8 XCDs round-robin (block b to XCD b % 8), so
// consecutive indices, whose wavefronts read the same element block's data,
// would otherwise sit in different L2s and fetch it from HBM once each.
__device__ __forceinline__ unsigned xcd_block()
{
    const unsigned b = blockIdx.x, nb = gridDim.x;
    const unsigned per = nb/8, rem = nb % 8, x = b % 8;
    return x*per + min(x, rem) + b/8;
}

// Element row of p at a uniform offset u (elements; scalar registers) plus a
// lane's byte offset: one 32-bit register addresses all rows of an array.
template <typename T>
__device__ __forceinline__ T &at(T *p, long u, unsigned lane)
{
    using C = typename std::conditional<std::is_const<T>::value, const char,
                                        char>::type;
    return *reinterpret_cast<T *>(reinterpret_cast<C *>(p + u) + lane);
}

// The same where p and u are uniform in a loop: the row's address is made
// opaque (scalar), or loop optimisation folds the lane's offset into a
// 64-bit vector address for every access.
template <typename T>
using GlobalRef = T __attribute__((address_space(1))) &;

template <typename T>
__device__ __forceinline__ GlobalRef<T> row_at(T *p, long u, unsigned lane)
{
    const uintptr_t q = reinterpret_cast<uintptr_t>(p + u);
    const uintptr_t lo = (unsigned)__builtin_amdgcn_readfirstlane((int)q);
    const uintptr_t hi = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(q >> 32));
    using B = char __attribute__((address_space(1)));
    using G = T __attribute__((address_space(1)));
    return *(G *)((B *)(hi << 32 | lo) + lane);
}

// A pointer read from memory, known to point to device memory (accesses
// through it are otherwise flat: they also occupy and wait for the LDS path).
template <typename T>
__device__ __forceinline__ T *global_ptr(T *p)
{
    using G = T __attribute__((address_space(1)));
    return (T *)(G *)p;
}

inline hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }

inline unsigned int cdiv(long a, long b) { return (unsigned int)((a + b - 1) / b); }

// Per-device address of the workspace-free reduction's scratch array
// (frhip_blasext.hip); frhip_init looks it up for its device.  Returns a
// hipError_t.
int red_scratch_init(int device);

}  // namespace frhip
