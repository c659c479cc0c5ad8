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

// Left-to-right sums of the w samples from x + e on, for e = 0 .. 3; reads
// x[0 .. reach4(w) - 1].
__device__ __forceinline__ int64_t reach4(int64_t w) { return ((w + 3) & ~3ll) + 4; }
__device__ __forceinline__ float4a window_sums4(const float* x, int64_t w) {
    float4a s = {0.0f, 0.0f, 0.0f, 0.0f};
    float4a a = *reinterpret_cast<const float4u*>(x);
    for (int64_t j = 0; j < w; j += 4) {
        const float4a b = *reinterpret_cast<const float4u*>(x + j + 4);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (j + i >= w) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += v[e + i];
        }
        a = b;
    }
    return s;
}
// The same for windows lo[e] .. hi[e] of a row of cols samples (hi < lo: no
// sample; lo non-decreasing, all inside the row otherwise).
__device__ __forceinline__ float4a window_sums4_clipped(const float* row, int64_t cols, const int64_t (&lo)[4],
                                                        const int64_t (&hi)[4]) {
    float4a s = {0.0f, 0.0f, 0.0f, 0.0f};
    const int64_t end = max(max(hi[0], hi[1]), max(hi[2], hi[3]));
    // positions from lo[0] on fit 32 bits: windows are at most 2^31 samples
    uint32_t l[4], h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const bool any = hi[e] >= lo[e];
        l[e] = any ? (uint32_t)(lo[e] - lo[0]) : 1u;
        h[e] = any ? (uint32_t)(hi[e] - lo[0]) : 0u;
    }
    auto add = [&](uint32_t j, const float4a& v) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = j + i >= l[e] && j + i <= h[e] ? s[e] + v[i] : s[e];
    };
    int64_t k = lo[0];
    for (; k <= end && k + 16 <= cols; k += 16) {
        float4a b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = *reinterpret_cast<const float4u*>(row + k + 4 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) add((uint32_t)(k - lo[0]) + 4 * q, b[q]);
    }
    for (; k <= end; k += 4) {  // the row's last samples
        float4a v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < cols) v[i] = row[k + i];
        add((uint32_t)(k - lo[0]), v);
    }
    return s;
}

}  // namespace
}  // namespace sps
