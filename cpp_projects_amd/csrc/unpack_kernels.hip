// unpack_kernels.hip -- 8-bit raw-voltage unpack into overlapping complex FFT
// blocks, the input side of the coherent front-end.
//
// Both layouts produce out[pol][fft][chan][bin] (complex float, re/im
// interleaved) for pol < npol / 2, fft < nfft, chan < nchan, bin < nbin, with
// sample isamp = bin + (nbin - 2 * noverlap) * fft - noverlap of the chunk
// (0 + 0i where isamp lies outside [0, nsamp)):
//   GUPPI (CDMT/Session_guppi_gpu.cu:116-140, unpack_guppi/kernel.cu:161-187):
//     in[chan][isamp][npol], pol p's (re, im) at components 2p, 2p + 1;
//   LOFAR (CDMT/Session_lofar_gpu.cu:144-175, unpack_guppi/kernel.cu:81-122):
//     in[component][isamp][chan], pol p's (re, im) in components 2p, 2p + 1.
// Samples are signed bytes, promoted exactly to float.  The work is pure
// byte-to-float streaming (each input byte read once per block it falls in,
// 8 output bytes per complex value), bounded by HBM bandwidth.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"

namespace sps {
namespace {

typedef float float4a __attribute__((ext_vector_type(4), aligned(16)));
typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ float byte_of(uint32_t w, int e) { return (float)(int8_t)((w >> (8 * e)) & 0xffu); }

// GUPPI: one lane per (chan, fft, bin), a lane reading the npol bytes of its
// sample: one by one, or as one word (two polarisations, 4-byte aligned input:
// 65535 bins, 64 channels, 4 blocks 91 us byte by byte, 81 so).  Output rows
// that are 16-byte aligned as well take two bins a lane, one 8-byte load and one
// 16-byte store per polarisation, kGuppiSteps of them in flight: 1.07 GB of
// blocks in 230 us, 298 with one bin a lane.
enum GuppiLane { kGuppiByte, kGuppiWord, kGuppiPair };
constexpr int kGuppiSteps = 4;

template <GuppiLane LANE>
__global__ void __launch_bounds__(kThreads) k_unpack_guppi(const int8_t* __restrict__ in, int64_t nsamp,
                                                           int noverlap, int nbin, int nfft, int npol, int nchan,
                                                           float2* __restrict__ out) {
    const int64_t ifft = blockIdx.y;
    const int64_t ichan = blockIdx.z;
    const int64_t base = (int64_t)(nbin - 2 * noverlap) * ifft - noverlap;  // bin 0's sample
    const int8_t* src = in + ichan * nsamp * npol;
    const int64_t plane = (int64_t)nfft * nchan * nbin;
    float2* dst = out + (ifft * nchan + ichan) * nbin;
    if constexpr (LANE == kGuppiPair) {
        const int64_t b0 = (int64_t)blockIdx.x * (2 * kThreads * kGuppiSteps) + 2 * threadIdx.x;
        u32x2u w[kGuppiSteps];
#pragma unroll
        for (int j = 0; j < kGuppiSteps; ++j) {
            const int64_t isamp = b0 + (int64_t)j * 2 * kThreads + base;
            w[j] = u32x2u{0u, 0u};
            if (b0 + (int64_t)j * 2 * kThreads < nbin) {
                if (isamp >= 0 && isamp + 1 < nsamp) {
                    w[j] = *reinterpret_cast<const u32x2u*>(src + 4 * isamp);
                } else {
                    if (isamp >= 0 && isamp < nsamp) w[j].x = *reinterpret_cast<const uint32_t*>(src + 4 * isamp);
                    if (isamp + 1 >= 0 && isamp + 1 < nsamp)
                        w[j].y = *reinterpret_cast<const uint32_t*>(src + 4 * isamp + 4);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kGuppiSteps; ++j) {
            const int64_t b = b0 + (int64_t)j * 2 * kThreads;
            if (b >= nbin) break;
            *reinterpret_cast<float4a*>(dst + b) =
                float4a{byte_of(w[j].x, 0), byte_of(w[j].x, 1), byte_of(w[j].y, 0), byte_of(w[j].y, 1)};
            *reinterpret_cast<float4a*>(dst + plane + b) =
                float4a{byte_of(w[j].x, 2), byte_of(w[j].x, 3), byte_of(w[j].y, 2), byte_of(w[j].y, 3)};
        }
    } else {
        const int64_t ibin = (int64_t)blockIdx.x * kThreads + threadIdx.x;
        if (ibin >= nbin) return;
        const int64_t isamp = ibin + base;
        const bool inside = isamp >= 0 && isamp < nsamp;
        src += (inside ? isamp : 0) * npol;
        if constexpr (LANE == kGuppiWord) {
            const uint32_t w = inside ? *reinterpret_cast<const uint32_t*>(src) : 0u;
            dst[ibin] = make_float2(byte_of(w, 0), byte_of(w, 1));
            dst[plane + ibin] = make_float2(byte_of(w, 2), byte_of(w, 3));
            return;
        }
        for (int p = 0; p < npol / 2; ++p) {
            float2 v = make_float2(0.0f, 0.0f);
            if (inside) v = make_float2((float)src[2 * p], (float)src[2 * p + 1]);
            dst[p * plane + ibin] = v;
        }
    }
}

// LOFAR: one block per (bins, channels, fft, pol) tile.  The tile's bytes are
// read along channels (coalesced), converted, transposed through LDS and
// written along bins (coalesced); the odd row length keeps the transposed
// reads free of bank conflicts.  A tile holds up to 64 channels in equal
// shares, and the fewer channels the more bins (64 to 256), so that a narrow
// band fills it: 20 channels, 35 MB of blocks, 22.6 us with 64 x 64 tiles for
// every band and 8-byte stores, 14.8 so.
constexpr int kUnpackTile = 64 * 65;  // complex values of the largest of the three tile shapes

// The bins of a tile are a template argument and a quad's index comes from a
// multiplication (`inv`, 65536 / quads rounded up: exact below 65536 / quads
// items), because divisions by run-time values had cost what odd rows, which
// keep the 8-byte stores, did not win back (64 channels x 101 bins x 400: 12.2
// us with fixed tiles, 14.1 with divisions, 12.2 so).
template <int TB>
__global__ void __launch_bounds__(kThreads) k_unpack_lofar(const int8_t* __restrict__ in, int64_t nsamp,
                                                           int noverlap, int nbin, int nfft, int nchan, int tc,
                                                           unsigned inv, float2* __restrict__ out) {
    constexpr unsigned tb = TB;
    __shared__ __attribute__((aligned(16))) float2 tile[kUnpackTile];  // [chan][bin], rows of tb + 1
    const int64_t bin0 = (int64_t)blockIdx.x * tb;
    const int64_t chan0 = (int64_t)blockIdx.y * tc;
    const int64_t ifft = blockIdx.z % (unsigned)nfft;
    const int64_t pol = blockIdx.z / (unsigned)nfft;
    const int8_t* re = in + (2 * pol) * nsamp * nchan;
    const int8_t* im = in + (2 * pol + 1) * nsamp * nchan;
    const int64_t step = nbin - 2 * noverlap;
    // four channels per item: one 4-byte load of each component when the
    // channel rows are 4-byte aligned and the four lie inside the band
    const bool words = (nchan & 3) == 0 && (reinterpret_cast<uintptr_t>(in) & 3) == 0;
    const unsigned quads = (unsigned)tc / 4;
    constexpr unsigned pitch = tb + 1;
    for (unsigned i = threadIdx.x; i < tb * quads; i += kThreads) {
        const unsigned b = (i * inv) >> 16, c = 4 * (i - b * quads);
        const int64_t ibin = bin0 + b, ichan = chan0 + c;
        const int64_t isamp = ibin + step * ifft - noverlap;
        const bool row = ibin < nbin && isamp >= 0 && isamp < nsamp;
        const int64_t k = isamp * nchan + ichan;
        if (words && row && ichan + 4 <= nchan) {
            const uint32_t wr = *reinterpret_cast<const uint32_t*>(re + k);
            const uint32_t wi = *reinterpret_cast<const uint32_t*>(im + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[(c + e) * pitch + b] = make_float2(byte_of(wr, e), byte_of(wi, e));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float2 v = make_float2(0.0f, 0.0f);
                if (row && ichan + e < nchan) v = make_float2((float)re[k + e], (float)im[k + e]);
                tile[(c + e) * pitch + b] = v;
            }
        }
    }
    __syncthreads();
    float2* dst = out + ((pol * nfft + ifft) * nchan) * (int64_t)nbin;
    if ((nbin & 1) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        constexpr unsigned half = tb / 2;
        for (unsigned i = threadIdx.x; i < (unsigned)tc * half; i += kThreads) {
            const unsigned c = i / half, b = 2 * (i % half);
            const int64_t ibin = bin0 + b, ichan = chan0 + c;
            if (ibin < nbin && ichan < nchan) {
                const float2 u = tile[c * pitch + b], v = tile[c * pitch + b + 1];
                *reinterpret_cast<float4a*>(dst + ichan * nbin + ibin) = float4a{u.x, u.y, v.x, v.y};
            }
        }
    } else {
        for (unsigned i = threadIdx.x; i < (unsigned)tc * tb; i += kThreads) {
            const unsigned c = i / tb, b = i % tb;
            const int64_t ibin = bin0 + b, ichan = chan0 + c;
            if (ibin < nbin && ichan < nchan) dst[ichan * nbin + ibin] = tile[c * pitch + b];
        }
    }
}

void check_unpack(int64_t nsamp, int noverlap, int nbin, int nfft, int npol, int nchan) {
    if (nsamp < 0 || noverlap < 0 || nbin < 1 || nfft < 1 || nchan < 1)
        throw Error(SPS_ERR_INVALID_ARGUMENT, "unpack sizes must be positive (nsamp, noverlap >= 0)");
    if (nbin <= 2 * noverlap) throw Error(SPS_ERR_INVALID_ARGUMENT, "nbin must exceed twice the overlap");
    if (npol != 2 && npol != 4) throw Error(SPS_ERR_INVALID_ARGUMENT, "npol must be 2 or 4 (re/im per polarisation)");
    if (nfft > 65535 || nchan > 65535) throw Error(SPS_ERR_INVALID_ARGUMENT, "nfft and nchan must be below 65536");
}

}  // namespace

void launch_unpack_guppi(const int8_t* in, int64_t nsamp, int noverlap, int nbin, int nfft, int npol, int nchan,
                         float* out, hipStream_t st) {
    check_unpack(nsamp, noverlap, nbin, nfft, npol, nchan);
    const bool words = npol == 4 && (reinterpret_cast<uintptr_t>(in) & 3) == 0;
    const bool pairs = words && (nbin & 1) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const int64_t bins = pairs ? 2 * kThreads * kGuppiSteps : kThreads;
    const dim3 grid((unsigned)ceil_div((int64_t)nbin, bins), (unsigned)nfft, (unsigned)nchan);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, in, nsamp, noverlap, nbin, nfft, npol, nchan,
                           reinterpret_cast<float2*>(out));
    };
    if (pairs) go(&k_unpack_guppi<kGuppiPair>);
    else if (words) go(&k_unpack_guppi<kGuppiWord>);
    else go(&k_unpack_guppi<kGuppiByte>);
    SPS_HIP(hipGetLastError());
}

void launch_unpack_lofar(const int8_t* in, int64_t nsamp, int noverlap, int nbin, int nfft, int npol, int nchan,
                         float* out, hipStream_t st) {
    check_unpack(nsamp, noverlap, nbin, nfft, npol, nchan);
    const int64_t z = (int64_t)nfft * (npol / 2);
    if (z > 65535) throw Error(SPS_ERR_INVALID_ARGUMENT, "nfft * polarisations must be below 65536");
    const int64_t ctiles = ceil_div((int64_t)nchan, (int64_t)64);
    const int tc = (int)(ceil_div(ceil_div((int64_t)nchan, ctiles), (int64_t)4) * 4);
    const int tb = tc > 32 ? 64 : (tc > 16 ? 128 : 256);
    const dim3 grid((unsigned)ceil_div((int64_t)nbin, (int64_t)tb), (unsigned)ceil_div((int64_t)nchan, (int64_t)tc),
                    (unsigned)z);
    const unsigned inv = (65536u + (unsigned)tc / 4 - 1) / ((unsigned)tc / 4);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, in, nsamp, noverlap, nbin, nfft, nchan, tc, inv,
                           reinterpret_cast<float2*>(out));
    };
    if (tb == 64) go(&k_unpack_lofar<64>);
    else if (tb == 128) go(&k_unpack_lofar<128>);
    else go(&k_unpack_lofar<256>);
    SPS_HIP(hipGetLastError());
}

}  // namespace sps
