// init_values.hpp -- device pieces shared by the FDMT kernels: the XCD-aware
// block order, vector types, and the normalised init values.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace sps {
namespace {

constexpr int kNumXcd = 8;

__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nblocks) {
    const uint32_t xcd = b % kNumXcd, k = b / kNumXcd;
    const uint32_t q = nblocks / kNumXcd, rem = nblocks % kNumXcd;
    return xcd * q + min(xcd, rem) + k;
}

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float4a __attribute__((ext_vector_type(4), aligned(16)));

// four bytes at any alignment (one load: the target's unaligned access mode)
typedef uint32_t u32u __attribute__((aligned(1)));

// One whole 16-byte LDS write (p 16-byte aligned; said so, or the compiler
// splits it into 4-byte pairs with the same strided pattern).
__device__ __forceinline__ void lds_store4(float* p, float4a v) {
    *static_cast<float4a*>(__builtin_assume_aligned(p, 16)) = v;
}

template <int IN_KIND>
__device__ __forceinline__ float4a unpack_chunk(uint32_t w8, const float4a& wf) {
    if constexpr (IN_KIND == 1) {
        float4a v;
        v.x = (float)(w8 & 0xffu);
        v.y = (float)((w8 >> 8) & 0xffu);
        v.z = (float)((w8 >> 16) & 0xffu);
        v.w = (float)(w8 >> 24);
        return v;
    } else {
        return wf;
    }
}

// (a - mu) / sigma correctly rounded for four samples, as div_rn computes it,
// with one branch for the rare operands outside its fast range
__device__ __forceinline__ float4a norm4(float4a v, float mu, float sg, float rsg) {
    const float a[4] = {v.x - mu, v.y - mu, v.z - mu, v.w - mu};
    float q[4];
    bool slow = !(sg >= 0x1p-60f && sg <= 0x1p60f);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float ax = fabsf(a[e]);
        slow = slow || !(ax >= 0x1p-60f && ax <= 0x1p60f);
        const float q0 = a[e] * rsg;
        const float r = fmaf(-q0, sg, a[e]);
        q[e] = fmaf(r, rsg, q0);
    }
    if (slow) {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = div_rn(a[e], sg, rsg);
    }
    return float4a{q[0], q[1], q[2], q[3]};
}

// 8-bit channels whose every normalised sample lies in a range where the
// init needs no operand checks.  For v = 0..255, a(v) = fl(v - mu) and
// x(v) = fl(a(v) / sigma) are non-decreasing in v and vanish only at v = mu,
// so |a| and |x| are smallest at the integers next to mu and largest at 0 or
// 255; checking those five samples checks all 256.  If sigma and every
// nonzero |a| lie in [2^-60, 2^60], the quotient's fast form q0 = a * rsg,
// q0 + rsg * (a - q0 * sigma) is the division (norm4's fast branch); +0 for
// a = +0, never -0.  If every nonzero |x| lies in [2^-60, 2^60] too, every
// init row value is +0 or between 2^-113 and 2^64 in magnitude: sums and
// integer multiples of values on the 2^-83 grid stay on it, so the dividend
// of the division by 3 (row 2) is +0 or at least 2^-83, row 2 at least
// 2^-85 (a float on the 2^-108 grid), the dividend of the division by 5
// (row 4) +0 or at least 2^-110.  The fast quotient by the constants 3 and 5
// is then exact without checks: it scales exactly with its operand's binade
// while every step stays normal, and tests/cpp/div_check.c tries every
// mantissa of one binade against both divisors.
__device__ __forceinline__ bool u8_init_plain(float mu, float sg) {
    if (!(sg >= 0x1p-60f && sg <= 0x1p60f) || !(fabsf(mu) <= 0x1p30f)) return false;
    const int f = (int)floorf(mu);
    const int cand[5] = {0, 255, f - 1, f, f + 1};
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int v = cand[i];
        if (v < 0 || v > 255) continue;
        const float a = (float)v - mu;
        if (a == 0.0f) continue;
        const float aa = fabsf(a), ax = fabsf(a / sg);
        ok = ok && aa >= 0x1p-60f && aa <= 0x1p60f && ax >= 0x1p-60f && ax <= 0x1p60f;
    }
    return ok;
}

}  // namespace
}  // namespace sps
