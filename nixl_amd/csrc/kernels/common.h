// Shared by the kernel translation units: error reporting for the C ABI and small device
// helpers.
#ifndef NIXL_AMD_KERNELS_COMMON_H
#define NIXL_AMD_KERNELS_COMMON_H

#include <hip/hip_runtime.h>

#include <string>

#include "nixl_amd_hip.h"

// Records `msg` as the calling thread's last error and returns `code`.
int
nixl_amd_fail(int code, const std::string &msg);

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return nixl_amd_fail(NIXL_AMD_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Makes `device` current for the calling thread for the lifetime of the object and puts the
// thread's previous device back afterwards: a library call must not leave the application on
// another GPU than it was on.
class DeviceScope {
public:
    explicit DeviceScope(int device) {
        int current = -1;
        if (hipGetDevice(&current) != hipSuccess) current = -1;
        if (current == device) {
            status_ = hipSuccess;
            return;
        }
        status_ = hipSetDevice(device);
        if (status_ == hipSuccess && current >= 0) previous_ = current;
    }

    ~DeviceScope() {
        if (previous_ >= 0) (void)hipSetDevice(previous_);
    }

    DeviceScope(const DeviceScope &) = delete;
    DeviceScope &
    operator=(const DeviceScope &) = delete;

    hipError_t
    status() const {
        return status_;
    }

private:
    int previous_ = -1;
    hipError_t status_ = hipSuccess;
};

constexpr int kWaveSize = 64;

__device__ __forceinline__ uint32_t
uniform(uint32_t v) {
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ uint64_t
uniform64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Sum of one 32-bit value per lane over the wave, or of 16-bit fields that do not overflow: in every lane.
__device__ __forceinline__ uint32_t
wave_sum_dpp(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0xb1, 0xf, 0xf, false); // quad_perm [1,0,3,2]
    x += __builtin_amdgcn_update_dpp(0u, x, 0x4e, 0xf, 0xf, false); // quad_perm [2,3,0,1]
    x += __builtin_amdgcn_update_dpp(0u, x, 0x124, 0xf, 0xf, false); // row_ror 4
    x += __builtin_amdgcn_update_dpp(0u, x, 0x128, 0xf, 0xf, false); // row_ror 8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false); // row_bcast 15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false); // row_bcast 31 into rows 2 and 3
    return __builtin_amdgcn_readlane(x, kWaveSize - 1);
}

// The same up to and with each lane.
__device__ __forceinline__ uint32_t
wave_scan_dpp(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xf, 0xf, false); // row_shr 1
    x += __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xf, 0xf, false); // row_shr 2
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xf, 0xf, false); // row_shr 4
    x += __builtin_amdgcn_update_dpp(0u, x, 0x118, 0xf, 0xf, false); // row_shr 8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false); // row_bcast 15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false); // row_bcast 31 into rows 2 and 3
    return x;
}

// Division by a number that the host knows: a multiplication and four more instructions in place of the 27
// of a division, each of which a wave waits 2.5 ns for before its first load (Granlund and Montgomery, "Division
// by invariant integers using multiplication", 1994; exact for every 32-bit dividend).
struct FastDiv {
    uint32_t divisor, mul, shift_1, shift_2;

    FastDiv() : FastDiv(1) {}

    explicit FastDiv(uint32_t d) : divisor(d) { // not 0
        int bits = 0; // 2^bits is the first power of two not below the divisor
        while (bits < 32 && (1ull << bits) < d)
            ++bits;
        mul = static_cast<uint32_t>((((1ull << bits) - d) << 32) / d + 1);
        shift_1 = bits > 0 ? 1 : 0;
        shift_2 = bits > 0 ? bits - 1 : 0;
    }

    __host__ __device__ __forceinline__ uint32_t
    quotient(uint32_t n) const {
        const uint32_t t = static_cast<uint32_t>((static_cast<uint64_t>(mul) * n) >> 32);
        return (t + ((n - t) >> shift_1)) >> shift_2;
    }

    __host__ __device__ __forceinline__ uint32_t
    quotient(uint32_t n, uint32_t &rest) const {
        const uint32_t q = quotient(n);
        rest = n - q * divisor;
        return q;
    }
};

#endif
