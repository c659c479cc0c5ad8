// sort_kernels.hip -- stable LSD radix sort, scans and candidate clustering.
//
// The clustering of Clusterization.cu:92-166,793-998 (per-group segmented
// sorts by mt, mdt, mwidth with gap splits) is expressed as three global
// stable sorts on composite keys (group id above the member, both at their
// actual widths), which visit the same groups in the same member order as a
// stable segmented sort.
#include "common.hpp"
#include "kernels.hpp"

namespace sps {

namespace {

constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;
constexpr int kMaxDigits = 8;
constexpr int kItemsPerThread = 8;
constexpr int kSortThreads = 512;
constexpr int kSortTile = kSortThreads * kItemsPerThread;  // items per tile of k_sort_pass
constexpr int kGroupTile = kThreads * kItemsPerThread;     // of k_cluster_groups
constexpr int kSmallThreads = 1024;                        // of k_sort_small
constexpr int kWave = 64;
constexpr int kWaves = kThreads / kWave;
static_assert(kThreads == kRadix, "one thread per digit");

// What tiles publish for the tiles after them, one word per tile and digit (or
// per tile): bits 63..62 say what it holds (1: the tile's own count, 2: the
// count of all tiles up to it), 61..56 the pass it belongs to, the rest the
// count.  Flag and count travel in one 64-bit atomic, so no fence is needed.
constexpr uint64_t kOwn = 1, kUpTo = 2;
__device__ __forceinline__ uint64_t tile_word(uint64_t what, uint32_t pass, uint64_t count) {
    return what << 62 | (uint64_t)pass << 56 | count;
}
__device__ __forceinline__ void publish(uint64_t* w, uint64_t v) {
    __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Sum of the counts of tiles 0 .. tile - 1 (words stride apart): the decoupled
// look-back of Merrill and Garland's single-pass scan (2016).  Tiles take
// their numbers from a counter as they start and publish their own counts
// before they look back, so every tile waited for is running or done and
// never waits for a later one.  Eight words are read at a time: with all
// tiles of a launch in flight the walk back is a chain of some sqrt(2 tiles)
// memory latencies, which was most of a pass (k_sort_pass over 576 tiles: 23.0 us with
// one word at a time, 20.3 with eight).
__device__ __forceinline__ uint64_t look_back(const uint64_t* words, int64_t tile, int64_t stride, uint32_t pass) {
    constexpr int kAhead = 8;
    uint64_t sum = 0;
    int64_t t = tile - 1;
    while (t >= 0) {
        uint64_t v[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            v[j] = __hip_atomic_load(words + (t >= j ? t - j : 0) * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool go = true;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            go = go && t >= 0 && (v[j] >> 62) != 0 && ((v[j] >> 56) & 63u) == pass;
            if (go) {
                sum += v[j] & (((uint64_t)1 << 56) - 1);
                t = (v[j] >> 62) == kUpTo ? -1 : t - 1;
            }
        }
    }
    return sum;
}
// The same for one word per tile, by a whole wave: 64 words at a time.
__device__ __forceinline__ uint32_t look_back_wave(const uint64_t* words, int64_t tile, uint32_t pass) {
    const int lane = (int)threadIdx.x & (kWave - 1);
    uint32_t sum = 0;
    int64_t t = tile - 1;
    while (t >= 0) {
        const uint64_t v = t >= lane ? __hip_atomic_load(words + (t - lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                     : tile_word(kUpTo, pass, 0);
        const bool ready = (v >> 62) != 0 && ((v >> 56) & 63u) == pass;
        const uint64_t wait = __ballot(!ready), upto = __ballot(ready && (v >> 62) == kUpTo);
        const int w = wait ? __builtin_ctzll(wait) : kWave, u = upto ? __builtin_ctzll(upto) : kWave;
        if (lane < w && lane <= u) sum += (uint32_t)v;
        t = u < w ? -1 : t - w;
    }
    for (int off = kWave / 2; off > 0; off >>= 1) sum += (uint32_t)__shfl_xor((int)sum, off);
    return sum;
}
__device__ __forceinline__ uint32_t take_tile(uint32_t* counter, uint32_t* sh) {
    if (threadIdx.x == 0) *sh = atomicAdd(counter, 1u);
    __syncthreads();
    return *sh;
}

// Counts of every digit of every pass, one read of the keys.  At most 256
// blocks, because their additions to a digit's count serialise; 1024 threads
// each to hide the LDS atomics (7.9 M keys of 64 bits, 5 digits: 88 us with
// 256 threads and one key in flight, 78 with eight, 46 so).
constexpr int kHistThreads = 1024;
template <typename K>
__global__ void __launch_bounds__(kHistThreads) k_sort_hist(const K* __restrict__ keys, int64_t n, int passes,
                                                        uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[kMaxDigits][kRadix];
    for (int i = (int)threadIdx.x; i < passes * kRadix; i += kHistThreads) h[i / kRadix][i % kRadix] = 0;
    __syncthreads();
    const int64_t step = (int64_t)gridDim.x * kHistThreads;
    const int lane = (int)threadIdx.x & (kWave - 1);
    constexpr int kAhead = 4;
    for (int64_t i0 = (int64_t)blockIdx.x * kHistThreads; i0 < n; i0 += kAhead * step) {  // block-uniform
        K k[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) k[j] = keys[min(i0 + j * step + (int64_t)threadIdx.x, n - 1)];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const bool in = i0 + j * step + (int64_t)threadIdx.x < n;
            const uint64_t on = __ballot(in);
            if (!on) break;  // wave-uniform
            for (int p = 0; p < passes; ++p) {
                const uint32_t d = (uint32_t)(k[j] >> (p * kRadixBits)) & (kRadix - 1);
                // sorted or clustered keys: one add for a wave that agrees
                const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
                if (__ballot(in && d == d0) == on) {
                    if (lane == 0) atomicAdd(&h[p][d0], (uint32_t)__popcll(on));
                } else if (in) {
                    atomicAdd(&h[p][d], 1u);
                }
            }
        }
    }
    __syncthreads();
    for (int i = (int)threadIdx.x; i < passes * kRadix; i += kHistThreads)
        if (h[i / kRadix][i % kRadix]) atomicAdd(&hist[i], h[i / kRadix][i % kRadix]);
}

// inclusive scan over the block (one value per thread), in LDS
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* sh) {
    const int lane = (int)threadIdx.x & (kWave - 1), w = (int)threadIdx.x / kWave;
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)v, off);
        if (lane >= off) v += o;
    }
    __syncthreads();
    if (lane == kWave - 1) sh[w] = v;
    __syncthreads();
    for (int k = 0; k < w; ++k) v += sh[k];
    return v;
}

// rank[j]: how many items of the wave before item j share its digit; the
// wave's counts of all digits end up in `counts` (LDS, cleared before).  Lane and j give
// item (wave * N + j) * 64 + lane of the tile's m; equal digits are found with
// 8 ballots.
template <typename K, int N>
__device__ __forceinline__ void rank_digits(const K (&k)[N], int first, int m, int shift, uint16_t* counts,
                                            uint16_t (&rank)[N]) {
    // (said to be in LDS: volatile accesses through a generic pointer stay flat
    // ones, which wait for global memory too; 30000 pairs 9.75 -> 9.16 us a digit)
    typedef volatile __attribute__((address_space(3))) uint16_t lds_u16;
    lds_u16* const wc = (lds_u16*)counts;
    const int lane = (int)threadIdx.x & (kWave - 1);
    const uint64_t below = lane == 0 ? 0ull : ~0ull >> (64 - lane);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const bool in = first + j * kWave + lane < m;
        const uint32_t d = (uint32_t)(k[j] >> shift) & (kRadix - 1);
        uint64_t peers = __ballot(in);
#pragma unroll
        for (int bit = 0; bit < kRadixBits; ++bit) {
            const uint64_t bal = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? bal : ~bal;
        }
        const uint32_t before = wc[d];  // read by all lanes before any of them adds
        __builtin_amdgcn_wave_barrier();
        const uint32_t r = (uint32_t)__popcll(peers & below);
        if (in && r == 0) wc[d] = (uint16_t)(before + (uint32_t)__popcll(peers));
        __builtin_amdgcn_wave_barrier();
        rank[j] = (uint16_t)(before + r);
    }
}

// Counts of the waves before each, in place; returns the tile's count (digits
// only: thread = digit).
template <int W>
__device__ __forceinline__ uint32_t sum_waves(uint16_t (*wcount)[kRadix]) {
    uint32_t total = 0;
    if (threadIdx.x < kRadix) {
        for (int q = 0; q < W; ++q) {
            const uint32_t c = wcount[q][threadIdx.x];
            wcount[q][threadIdx.x] = (uint16_t)total;
            total += c;
        }
    }
    return total;
}

// LDS of a block that sorts up to 1024 N pairs by itself.
template <typename K, int N>
struct SmallSort {
    static constexpr int kW = kSmallThreads / kWave;
    uint16_t wcount[kW][kRadix];
    uint16_t start[kRadix];
    uint32_t scan[kW];
    K items[kSmallThreads * N];
};

// Sorts the block's n pairs k, v (lane, wave and j give item (wave * N + j) *
// 64 + lane) by `passes` digits: the pairs stay in registers and change places
// through LDS.
template <typename K, int N>
__device__ __forceinline__ void small_sort(SmallSort<K, N>& s, K (&k)[N], uint32_t (&v)[N], int n, int passes) {
    constexpr int kW = SmallSort<K, N>::kW;
    uint32_t* const lv = reinterpret_cast<uint32_t*>(s.items);
    const int tid = (int)threadIdx.x;
    const int w = tid / kWave, first = w * N * kWave, at0 = first + (tid & (kWave - 1));
    uint16_t rank[N];
    for (int p = 0; p < passes; ++p) {
        const int shift = p * kRadixBits;
        for (int i = tid; i < kW * kRadix; i += kSmallThreads) s.wcount[i / kRadix][i % kRadix] = 0;
        __syncthreads();
        rank_digits<K, N>(k, first, n, shift, s.wcount[w], rank);
        __syncthreads();
        const uint32_t total = sum_waves<kW>(s.wcount);
        const uint32_t own = block_scan(total, s.scan) - total;
        if (tid < kRadix) s.start[tid] = (uint16_t)own;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (at0 + j * kWave >= n) continue;
            const uint32_t d = (uint32_t)(k[j] >> shift) & (kRadix - 1);
            rank[j] = (uint16_t)(s.start[d] + s.wcount[w][d] + rank[j]);
            s.items[rank[j]] = k[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (at0 + j * kWave < n) k[j] = s.items[at0 + j * kWave];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (at0 + j * kWave < n) lv[rank[j]] = v[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (at0 + j * kWave < n) v[j] = lv[at0 + j * kWave];
    }
}

// Every digit of a sort of at most 1024 N pairs, by one block, in place: one
// launch, and no digit waits for memory.  Bound by the chain of barriers (7201
// pairs of 4 digits: 22 us; a launch per digit, their counts and a fill: 42).
template <typename K, int N>
__global__ void __launch_bounds__(kSmallThreads) k_sort_small(K* __restrict__ keys, uint32_t* __restrict__ vals, int n,
                                                              int passes) {
    __shared__ SmallSort<K, N> s;
    const int at0 = (int)threadIdx.x / kWave * N * kWave + ((int)threadIdx.x & (kWave - 1));
    K k[N];
    uint32_t v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = at0 + j * kWave;
        k[j] = i < n ? keys[i] : (K)0;
        v[j] = i < n ? vals[i] : 0u;
    }
    small_sort<K, N>(s, k, v, n, passes);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = at0 + j * kWave;
        if (i < n) {
            keys[i] = k[j];
            vals[i] = v[j];
        }
    }
}

// One digit of a stable LSD sort, one launch: a tile ranks its items by digit,
// waves combined through their LDS counts, looks back for the counts of the
// tiles before it, and writes its items digit by digit from LDS, keys and
// values one after the other through the same buffer.  Bound by the scattered
// writes (runs of tile / 256 items), the words and the tile counter, all of
// which a larger tile thins out: 17.2 us at 1.18 M pairs of 8 bytes with 4096
// items, 20.3 with 2048 (1024 threads, 8192 items: 17.2, but 11.4 instead of
// 9.4 at 30000 pairs); with one launch for the counts, three for their scans
// and one to scatter a digit took 33 us.
template <typename K, int T>
__global__ void __launch_bounds__(T) k_sort_pass(const K* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                 int64_t n, int pass, const uint32_t* __restrict__ hist,
                                                 uint64_t* __restrict__ words, uint32_t* __restrict__ counters,
                                                 K* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
    constexpr int kTile = T * kItemsPerThread, kW = T / kWave;
    __shared__ uint16_t wcount[kW][kRadix];
    __shared__ uint16_t start[kRadix];  // the tile's first item of a digit, in its LDS order
    __shared__ uint32_t place[kRadix];  // output position of that item, less start
    __shared__ uint32_t scan[kW];
    __shared__ uint32_t tile_sh;
    __shared__ K items[kTile];
    const int tid = (int)threadIdx.x;
    const int lane = tid & (kWave - 1), w = tid / kWave;
    for (int i = tid; i < kW * kRadix; i += T) wcount[i / kRadix][i % kRadix] = 0;
    const int64_t tile = take_tile(&counters[pass], &tile_sh);
    const int64_t b0 = tile * kTile;
    const int m = (int)min((int64_t)kTile, n - b0);
    const int shift = pass * kRadixBits;
    K k[kItemsPerThread];
    uint32_t v[kItemsPerThread];
    uint16_t rank[kItemsPerThread];
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j) {
        const int i = (w * kItemsPerThread + j) * kWave + lane;
        k[j] = i < m ? keys[b0 + i] : (K)0;
        v[j] = i < m ? vals[b0 + i] : 0u;
    }
    rank_digits<K, kItemsPerThread>(k, w * kItemsPerThread * kWave, m, shift, wcount[w], rank);
    __syncthreads();
    const uint32_t total = sum_waves<kW>(wcount);
    uint32_t first = 0;
    if (tid < kRadix) {  // thread = digit
        publish(&words[tile * kRadix + tid], tile_word(tile == 0 ? kUpTo : kOwn, (uint32_t)pass + 1, total));
        first = hist[tid];
    }
    const uint32_t own = block_scan(total, scan) - total;  // (threads past the digits add nothing)
    first = block_scan(first, scan) - first;               // of the digit, over all items
    if (tid < kRadix) {
        start[tid] = (uint16_t)own;
        if (tile > 0) {
            const uint64_t before = look_back(words + tid, tile, kRadix, (uint32_t)pass + 1);
            publish(&words[tile * kRadix + tid], tile_word(kUpTo, (uint32_t)pass + 1, before + total));
            first += (uint32_t)before;
        }
        place[tid] = first - own;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j) {
        if ((w * kItemsPerThread + j) * kWave + lane >= m) continue;
        const uint32_t d = (uint32_t)(k[j] >> shift) & (kRadix - 1);
        rank[j] = (uint16_t)(start[d] + wcount[w][d] + rank[j]);
        items[rank[j]] = k[j];
    }
    __syncthreads();
    uint32_t at[kItemsPerThread];
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j) {
        const int i = j * T + tid;
        if (i >= m) continue;
        const K kk = items[i];
        at[j] = place[(uint32_t)(kk >> shift) & (kRadix - 1)] + (uint32_t)i;
        keys_out[at[j]] = kk;
    }
    __syncthreads();
    uint32_t* const lv = reinterpret_cast<uint32_t*>(items);
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j)
        if ((w * kItemsPerThread + j) * kWave + lane < m) lv[rank[j]] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j)
        if (j * T + tid < m) vals_out[at[j]] = lv[j * T + tid];
}

// ---- scan: inclusive, uint32, blocks of 1024 items (4 per thread) ----
constexpr int kScanItems = 4;
constexpr int kScanBlock = kThreads * kScanItems;

// exclusive prefix of v over the block (Hillis-Steele over the thread
// values; the exclusive value is the previous thread's inclusive one, so no
// subtraction enters a float scan)
template <typename T>
__device__ T block_excl_scan(T v, T* sh, T* total) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kThreads; off <<= 1) {
        const T add = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : T(0);
        __syncthreads();
        sh[threadIdx.x] += add;
        __syncthreads();
    }
    const T excl = threadIdx.x > 0 ? sh[threadIdx.x - 1] : T(0);
    *total = sh[kThreads - 1];
    __syncthreads();
    return excl;
}

template <typename T>
__global__ void __launch_bounds__(kThreads) k_scan_local(T* __restrict__ data, int64_t n, T* __restrict__ block_sums) {
    __shared__ T sh[kThreads];
    const int64_t base = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanItems;
    T x[kScanItems];
    T s = T(0);
    for (int e = 0; e < kScanItems; ++e) {
        x[e] = (base + e < n) ? data[base + e] : T(0);
        s += x[e];
    }
    T total;
    T pre = block_excl_scan<T>(s, sh, &total);
    for (int e = 0; e < kScanItems; ++e) {
        pre += x[e];
        if (base + e < n) data[base + e] = pre;
    }
    if (threadIdx.x == 0 && block_sums) block_sums[blockIdx.x] = total;
}

template <typename T>
__global__ void __launch_bounds__(kThreads) k_scan_add(T* __restrict__ data, int64_t n,
                                                       const T* __restrict__ block_prefix) {
    if (blockIdx.x == 0) return;
    const T add = block_prefix[blockIdx.x - 1];
    const int64_t base = (int64_t)blockIdx.x * kScanBlock;
    for (int e = threadIdx.x; e < kScanBlock; e += kThreads)
        if (base + e < n) data[base + e] += add;
}

// ---- candidates ----
__device__ __forceinline__ uint32_t ord_i32(int32_t v) { return (uint32_t)v ^ 0x80000000u; }
__device__ __forceinline__ uint32_t ord_f32(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

template <typename K>
__global__ void k_cand_keys(const CandD* __restrict__ c, int64_t n, int bits_t, int bits_w, K* __restrict__ keys,
                            uint32_t* __restrict__ vals, uint64_t* __restrict__ scratch, int64_t clear) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < clear) scratch[i] = 0;
    if (i >= n) return;
    const CandD x = c[i];
    keys[i] = (K)(((uint64_t)(uint32_t)x.mdt << (bits_t + bits_w)) | ((uint64_t)(uint32_t)x.mt << bits_w) |
                  (uint64_t)(uint32_t)x.mwidth);
    vals[i] = __float_as_uint(x.msnr);
}

template <typename K>
__global__ void k_cand_from_keys(const K* __restrict__ keys, const uint32_t* __restrict__ vals, int64_t n, int bits_t,
                                 int bits_w, CandD* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const uint64_t k = keys[i];
    CandD x;
    x.mwidth = (int32_t)(k & ((1ull << bits_w) - 1));
    x.mt = (int32_t)((k >> bits_w) & ((1ull << bits_t) - 1));
    x.mdt = (int32_t)(k >> (bits_t + bits_w));
    x.msnr = __uint_as_float(vals[i]);
    out[i] = x;
}

__device__ __forceinline__ int32_t member_of(const CandD& c, int m) { return m == 0 ? c.mt : (m == 1 ? c.mdt : c.mwidth); }

// ranges[2 m], ranges[2 m + 1]: the smallest and largest ord(member m), from
// {0xffffffff, 0} on.  One atomic per block and bound, and only where it moves
// it: the atomics on this one line are what a launch waits for (1.18 M
// candidates: 145 us with one per wave of 512 blocks, 10 us so).
__global__ void __launch_bounds__(kThreads) k_cand_ranges(const CandD* __restrict__ c, int64_t n,
                                                          uint32_t* __restrict__ ranges) {
    __shared__ uint32_t sh[kWaves][6];
    uint32_t lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
#pragma unroll 4
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        const CandD x = c[i];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const uint32_t o = ord_i32(member_of(x, m));
            lo[m] = min(lo[m], o);
            hi[m] = max(hi[m], o);
        }
    }
    const int lane = (int)threadIdx.x & (kWave - 1), w = (int)threadIdx.x / kWave;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        for (int off = kWave / 2; off > 0; off >>= 1) {
            lo[m] = min(lo[m], (uint32_t)__shfl_xor((int)lo[m], off));
            hi[m] = max(hi[m], (uint32_t)__shfl_xor((int)hi[m], off));
        }
        if (lane == 0) {
            sh[w][2 * m] = lo[m];
            sh[w][2 * m + 1] = hi[m];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        uint32_t v = sh[0][threadIdx.x];
        const bool low = (threadIdx.x & 1) == 0;
        for (int q = 1; q < kWaves; ++q) v = low ? min(v, sh[q][threadIdx.x]) : max(v, sh[q][threadIdx.x]);
        uint32_t* at = ranges + threadIdx.x;
        const uint32_t old = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (low && v < old) atomicMin(at, v);
        if (!low && v > old) atomicMax(at, v);
    }
}

// keys[i] = group[i] << bits | (ord(member(c[perm[i]])) - base), vals[i] =
// perm[i] (perm, group: null for the candidates' own order in one group)
template <typename K>
__global__ void k_cluster_keys(const CandD* __restrict__ c, const uint32_t* __restrict__ perm,
                               const uint32_t* __restrict__ group, int64_t n, int member, uint32_t base, int bits,
                               K* __restrict__ keys, uint32_t* __restrict__ vals, uint64_t* __restrict__ scratch,
                               int64_t clear) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < clear) scratch[i] = 0;
    if (i >= n) return;
    const uint32_t p = perm ? perm[i] : (uint32_t)i;
    const uint64_t g = group ? (uint64_t)group[i] : 0ull;
    keys[i] = (K)((g << bits) | (uint64_t)(ord_i32(member_of(c[p], member)) - base));
    vals[i] = p;
}

// flag[i] = 1 where a new group starts: first item, another parent group, or
// a member gap larger than the bin (Clusterization.cu:854-893,930-998), and
// group[i], their inclusive sum, in one launch (tiles as in k_sort_pass).
template <typename K>
__global__ void __launch_bounds__(kThreads) k_cluster_groups(const K* __restrict__ keys, int64_t n, int bits,
                                                             const int32_t* __restrict__ bins, int level,
                                                             uint64_t* __restrict__ words,
                                                             uint32_t* __restrict__ counter,
                                                             uint32_t* __restrict__ flags,
                                                             uint32_t* __restrict__ group) {
    __shared__ uint32_t scan[kWaves];
    __shared__ uint32_t tile_sh, before_sh;
    const int64_t tile = take_tile(counter, &tile_sh);
    const int64_t i0 = tile * kGroupTile + (int64_t)threadIdx.x * kItemsPerThread;
    const int64_t bin = bins[level];
    const uint64_t mask = ((uint64_t)1 << bits) - 1;
    uint32_t f[kItemsPerThread], sum = 0;
    const bool whole = i0 + kItemsPerThread <= n;  // (keys, flags and group are whole allocations: aligned)
    K k[kItemsPerThread];
    if (whole) {
        constexpr int kVec = 16 / sizeof(K);
        typedef K vec __attribute__((ext_vector_type(kVec)));
#pragma unroll
        for (int j = 0; j < kItemsPerThread; j += kVec) {
            const vec x = *reinterpret_cast<const vec*>(keys + i0 + j);
#pragma unroll
            for (int e = 0; e < kVec; ++e) k[j + e] = x[e];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kItemsPerThread; ++j) k[j] = i0 + j < n ? keys[i0 + j] : (K)0;
    }
    uint64_t a = i0 > 0 && i0 <= n ? (uint64_t)keys[i0 - 1] : 0ull;
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j) {
        const int64_t i = i0 + j;
        const uint64_t b = (uint64_t)k[j];
        f[j] = 0;
        if (i < n) {
            f[j] = 1u;
            if (i > 0 && (a >> bits) == (b >> bits)) f[j] = (int64_t)((b & mask) - (a & mask)) > bin ? 1u : 0u;
        }
        sum += f[j];
        a = b;
    }
    const uint32_t upto = block_scan(sum, scan);
    if (threadIdx.x >= kThreads - kWave) {  // the last wave: its last lane holds the tile's count
        const bool last = threadIdx.x == kThreads - 1;
        if (last) publish(&words[tile], tile_word(tile == 0 ? kUpTo : kOwn, 1, upto));
        const uint32_t before = look_back_wave(words, tile, 1);
        if (last) {
            if (tile > 0) publish(&words[tile], tile_word(kUpTo, 1, (uint64_t)before + upto));
            before_sh = before;
        }
    }
    __syncthreads();
    uint32_t g[kItemsPerThread], at = before_sh + upto - sum;
#pragma unroll
    for (int j = 0; j < kItemsPerThread; ++j) g[j] = at += f[j];
    if (whole) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < kItemsPerThread; j += 4) {
            *reinterpret_cast<u32x4*>(flags + i0 + j) = u32x4{f[j], f[j + 1], f[j + 2], f[j + 3]};
            *reinterpret_cast<u32x4*>(group + i0 + j) = u32x4{g[j], g[j + 1], g[j + 2], g[j + 3]};
        }
    } else {
#pragma unroll
        for (int j = 0; j < kItemsPerThread; ++j) {
            if (i0 + j < n) {
                flags[i0 + j] = f[j];
                group[i0 + j] = g[j];
            }
        }
    }
}

// The three levels of a clustering of at most 1024 N candidates by one block:
// member ranges, keys, sorts, group starts and ids, as the launches above take
// them in up to 17 and a read back (7201 candidates: 120 us of kernels and
// their gaps, 48 so).  perm, flags and group as there; info: {smallest, largest
// ord(mt), groups}.
template <int N>
__global__ void __launch_bounds__(kSmallThreads) k_cluster_small(const CandD* __restrict__ c, int n,
                                                                 const int32_t* __restrict__ bins,
                                                                 uint32_t* __restrict__ perm,
                                                                 uint32_t* __restrict__ flags,
                                                                 uint32_t* __restrict__ group,
                                                                 uint32_t* __restrict__ info) {
    using Sort = SmallSort<uint64_t, N>;
    __shared__ Sort s;
    __shared__ uint32_t lo_sh[Sort::kW], hi_sh[Sort::kW], cnt_sh[Sort::kW];
    const int tid = (int)threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
    const int at0 = w * N * kWave + lane;
    const uint64_t upto = ~0ull >> (63 - lane);
    uint64_t k[N];
    uint32_t v[N], g[N], f[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        v[j] = (uint32_t)(at0 + j * kWave);
        g[j] = 0;
        f[j] = 0;
    }
    uint32_t ng = 0;  // groups of the level before (none: one group, id 0)
    for (int level = 0; level < 3; ++level) {
        uint32_t o[N], lo = 0xffffffffu, hi = 0u;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            o[j] = 0;
            if (at0 + j * kWave < n) {
                o[j] = ord_i32(member_of(c[v[j]], level));
                lo = min(lo, o[j]);
                hi = max(hi, o[j]);
            }
        }
        for (int off = kWave / 2; off > 0; off >>= 1) {
            lo = min(lo, (uint32_t)__shfl_xor((int)lo, off));
            hi = max(hi, (uint32_t)__shfl_xor((int)hi, off));
        }
        if (lane == 0) {
            lo_sh[w] = lo;
            hi_sh[w] = hi;
        }
        __syncthreads();
        for (int q = 0; q < Sort::kW; ++q) {
            lo = min(lo, lo_sh[q]);
            hi = max(hi, hi_sh[q]);
        }
        if (level == 0 && tid == 0) {
            info[0] = lo;
            info[1] = hi;
        }
        const int bits = hi > lo ? 32 - __clz((int)(hi - lo)) : 0;
        const int all = bits + (ng ? 32 - __clz((int)ng) : 0);
#pragma unroll
        for (int j = 0; j < N; ++j) k[j] = (uint64_t)g[j] << bits | (uint64_t)(o[j] - lo);
        small_sort<uint64_t, N>(s, k, v, n, (all + kRadixBits - 1) / kRadixBits);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (at0 + j * kWave < n) s.items[at0 + j * kWave] = k[j];
        __syncthreads();
        const int64_t bin = bins[level];
        const uint64_t mask = ((uint64_t)1 << bits) - 1;
        uint32_t mine = 0;  // group starts of the wave's items before and at this one
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int i = at0 + j * kWave;
            bool start = false;
            if (i < n) {
                start = true;
                if (i > 0) {
                    const uint64_t a = s.items[i - 1];
                    if (a >> bits == k[j] >> bits) start = (int64_t)((k[j] & mask) - (a & mask)) > bin;
                }
            }
            const uint64_t m = __ballot(start);
            f[j] = start ? 1u : 0u;
            g[j] = mine + (uint32_t)__popcll(m & upto);
            mine += (uint32_t)__popcll(m);
        }
        if (lane == 0) cnt_sh[w] = mine;
        __syncthreads();
        uint32_t before = 0;
        ng = 0;
        for (int q = 0; q < Sort::kW; ++q) {
            if (q < w) before += cnt_sh[q];
            ng += cnt_sh[q];
        }
#pragma unroll
        for (int j = 0; j < N; ++j) g[j] += before;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = at0 + j * kWave;
        if (i < n) {
            perm[i] = v[j];
            flags[i] = f[j];
            group[i] = g[j];
        }
    }
    if (tid == 0) info[2] = ng;
}

// gid = inclusive scan of flags (1-based group id, so non-decreasing); best[g]
// = max of (ord(msnr) << 32 | ~index) -> max S/N, ties to the lowest index;
// start[g] = first sorted position of group g.
// One atomicMax per candidate serialises where a few groups hold them all (a
// bright pulse: 1.18 M candidates in 15 groups took 11.2 ms).  A wave takes
// kDelItems consecutive candidates and keeps each lane's running best while
// all 64 lanes see one group; it reduces over the lanes only when the group
// ends, so a long group costs one atomic per wave.  64 candidates that span
// several groups take a segmented maximum over the lanes and one atomic per
// group among them.
constexpr int kDelItems = 1024;

__device__ __forceinline__ unsigned long long shfl_up_u64(unsigned long long v, int off) {
    return ((unsigned long long)(uint32_t)__shfl_up((int)(v >> 32), off) << 32) | (uint32_t)__shfl_up((int)v, off);
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const unsigned long long o =
            ((unsigned long long)(uint32_t)__shfl_xor((int)(v >> 32), off) << 32) | (uint32_t)__shfl_xor((int)v, off);
        v = o > v ? o : v;
    }
    return v;
}

__global__ void __launch_bounds__(kThreads) k_cluster_delegates(const CandD* __restrict__ c,
                                                                const uint32_t* __restrict__ perm,
                                                                const uint32_t* __restrict__ gid,
                                                                const uint32_t* __restrict__ flags, int64_t n,
                                                                unsigned long long* __restrict__ best,
                                                                uint32_t* __restrict__ start) {
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int64_t w = (int64_t)blockIdx.x * kWaves + ((int)threadIdx.x >> 6);
    const int64_t i0 = w * kDelItems, i1 = min(n, i0 + kDelItems);
    uint32_t cur = 0;                // group the lanes' bests belong to (0: none)
    unsigned long long mine = 0ull;  // this lane's best of it
    auto flush = [&]() {
        if (cur == 0) return;  // wave-uniform
        const unsigned long long m = wave_max_u64(mine);
        if (lane == 0) atomicMax(&best[cur - 1u], m);
        cur = 0;
        mine = 0ull;
    };
    for (int64_t b = i0; b < i1; b += kWave) {  // wave-uniform
        const int64_t i = b + lane;
        const bool in = i < i1;
        const uint32_t g = in ? gid[i] : 0u;
        unsigned long long key = 0ull;
        if (in) {
            const uint32_t p = perm[i];
            key = ((unsigned long long)ord_f32(c[p].msnr) << 32) | (unsigned long long)(0xffffffffu - p);
            if (flags[i]) start[g - 1u] = (uint32_t)i;
        }
        const uint32_t g0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)g);
        if (__ballot(g == g0 || !in) == ~0ull) {  // one group (lane 0 is always in range)
            if (g0 != cur) {
                flush();
                cur = g0;
            }
            mine = key > mine ? key : mine;
            continue;
        }
        flush();
        // segmented inclusive maximum: groups are runs of lanes
        for (int off = 1; off < kWave; off <<= 1) {
            const uint32_t og = (uint32_t)__shfl_up((int)g, off);
            const unsigned long long ok = shfl_up_u64(key, off);
            if (lane >= off && og == g && ok > key) key = ok;
        }
        const uint32_t gn = (uint32_t)__shfl_down((int)g, 1);
        if (in && (lane == kWave - 1 || gn != g)) atomicMax(&best[g - 1u], key);
    }
    flush();
}

// keys[g] = ord(mt of group g's delegate) - base: a stable sort of them in
// group order sorts by (mt, group)
__global__ void k_delegate_keys(const CandD* __restrict__ c, const unsigned long long* __restrict__ best, int64_t ng,
                                uint32_t base, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                uint64_t* __restrict__ scratch, int64_t clear) {
    const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (g < clear) scratch[g] = 0;
    if (g >= ng) return;
    const uint32_t d = 0xffffffffu - (uint32_t)(best[g] & 0xffffffffull);
    keys[g] = ord_i32(c[d].mt) - base;
    vals[g] = (uint32_t)g;
}

__global__ void k_delegate_out(const unsigned long long* __restrict__ best, const uint32_t* __restrict__ start,
                               const uint32_t* __restrict__ order, int64_t ng, int64_t n,
                               int32_t* __restrict__ delegates, int64_t* __restrict__ sizes) {
    const int64_t j = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (j >= ng) return;
    const uint32_t g = order[j];
    delegates[j] = (int32_t)(0xffffffffu - (uint32_t)(best[g] & 0xffffffffull));
    const int64_t end = (g + 1 < (uint64_t)ng) ? (int64_t)start[g + 1] : n;
    sizes[j] = end - (int64_t)start[g];
}

__global__ void k_pack_delegates(const CandD* __restrict__ c, const int32_t* __restrict__ del,
                                 const int64_t* __restrict__ size, int64_t ng, DelegateD* __restrict__ out) {
    const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (g >= ng) return;
    out[g] = DelegateD{c[del[g]], size[g], del[g], 0};
}

__global__ void k_fill_u64(unsigned long long* v, int64_t n, unsigned long long val) {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n) v[i] = val;
}

inline uint32_t grid1(int64_t n) { return (uint32_t)ceil_div(n > 0 ? n : 1, kThreads); }

// select_delegates (select_delegates.cu:16-51,62-125) over caller-provided
// groups: group g is positions [begin[g], begin[g+1]) (the last ends at
// nidx) of the index array; its delegate is the candidate index there with
// the largest msnr, the first such position on ties -- the rule of
// thrust::max_element with a less-than comparator, which also keeps a NaN
// found at the group's first position.  One wave per group.
__global__ void __launch_bounds__(64) k_select_delegates(const CandD* __restrict__ c, const int32_t* __restrict__ idx,
                                                         int64_t nidx, const int32_t* __restrict__ begin,
                                                         int64_t ngroups, int32_t* __restrict__ out) {
    const int64_t g = blockIdx.x;
    const int64_t b = begin[g];
    const int64_t e = g + 1 < ngroups ? (int64_t)begin[g + 1] : nidx;
    if (b >= e) {
        if (threadIdx.x == 0) out[g] = -1;
        return;
    }
    const float first = c[idx[b]].msnr;
    if (!(first == first)) {
        if (threadIdx.x == 0) out[g] = idx[b];
        return;
    }
    float bv = first;
    int64_t bp = b;
    for (int64_t p = b + threadIdx.x; p < e; p += 64) {
        const float v = c[idx[p]].msnr;
        if (v > bv || (v == bv && p < bp)) {
            bv = v;
            bp = p;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_down(bv, off);
        const int64_t op = __shfl_down(bp, off);
        if (ov > bv || (ov == bv && op < bp)) {
            bv = ov;
            bp = op;
        }
    }
    if (threadIdx.x == 0) out[g] = idx[bp];
}

}  // namespace

// ---------------------------------------------------------------------------
int64_t scan_scratch_entries(int64_t n) {
    int64_t tot = 0;
    for (int64_t m = ceil_div(n, kScanBlock); m > 1; m = ceil_div(m, kScanBlock)) tot += m;
    return tot + 1;
}

template <typename T>
static void scan_inclusive(T* data, int64_t n, T* scratch, hipStream_t st) {
    if (n <= 0) return;
    const int64_t nb = ceil_div(n, kScanBlock);
    if (nb > 0x7fffffffLL) throw Error(SPS_ERR_INVALID_ARGUMENT, "scan too long");
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_local<T>, dim3(1), dim3(kThreads), 0, st, data, n, (T*)nullptr);
        SPS_HIP(hipGetLastError());
        return;
    }
    T* sums = scratch;
    hipLaunchKernelGGL(k_scan_local<T>, dim3((uint32_t)nb), dim3(kThreads), 0, st, data, n, sums);
    scan_inclusive<T>(sums, nb, scratch + nb, st);
    hipLaunchKernelGGL(k_scan_add<T>, dim3((uint32_t)nb), dim3(kThreads), 0, st, data, n, (const T*)sums);
    SPS_HIP(hipGetLastError());
}

void scan_inclusive_u32(uint32_t* data, int64_t n, uint32_t* scratch, hipStream_t st) {
    scan_inclusive<uint32_t>(data, n, scratch, st);
}

void scan_inclusive_f32(float* data, int64_t n, float* scratch, hipStream_t st) {
    scan_inclusive<float>(data, n, scratch, st);
}

// ---- sort ----
namespace {
// scratch of a sort: tile counters per pass, digit counts per pass, tile words
struct SortScratch {
    uint32_t *counters, *hist;
    uint64_t* words;
    int64_t clear;  // 8-byte words to clear before the first pass
};
SortScratch sort_scratch(void* p, int64_t n) {
    SortScratch s;
    s.counters = static_cast<uint32_t*>(p);
    s.hist = s.counters + 16;
    s.words = reinterpret_cast<uint64_t*>(s.hist + kMaxDigits * kRadix);
    s.clear = (16 + kMaxDigits * kRadix) / 2 + ceil_div(n, (int64_t)kSortTile) * kRadix;  // (no fewer than group tiles)
    return s;
}
}  // namespace

// 8-byte words that the launch making n keys clears (fewer than its n
// threads); none where one block sorts
static int64_t sort_clear(int64_t n) { return n <= 8 * kSmallThreads ? 0 : sort_scratch(nullptr, n).clear; }

size_t sort_scratch_bytes(int64_t n) { return 8 * (size_t)sort_scratch(nullptr, n > 0 ? n : 1).clear; }

template <typename K>
bool radix_sort_pairs(K* keys, uint32_t* vals, K* keys_tmp, uint32_t* vals_tmp, int64_t n, int nbits, void* scratch,
                      hipStream_t st) {
    if (n <= 1 || nbits <= 0) return false;
    if (n > 0xffffffffLL) throw Error(SPS_ERR_INVALID_ARGUMENT, "too many items to sort");
    const int passes = (nbits + kRadixBits - 1) / kRadixBits;
    if (passes > kMaxDigits || nbits > (int)(8 * sizeof(K))) throw Error(SPS_ERR_INVALID_ARGUMENT, "sort key too wide");
    if (n <= 8 * kSmallThreads) {
        // one block for all digits: 7201 pairs of 4 digits take 22 us and 1
        // launch, digit by digit 42 and 6; past 8192 the pairs leave the registers
        if (n <= kSmallThreads)
            hipLaunchKernelGGL((k_sort_small<K, 1>), dim3(1), dim3(kSmallThreads), 0, st, keys, vals, (int)n, passes);
        else
            hipLaunchKernelGGL((k_sort_small<K, 8>), dim3(1), dim3(kSmallThreads), 0, st, keys, vals, (int)n, passes);
        SPS_HIP(hipGetLastError());
        return false;
    }
    const SortScratch s = sort_scratch(scratch, n);
    const uint32_t tiles = (uint32_t)ceil_div(n, (int64_t)kSortTile);
    const uint32_t hb = (uint32_t)ceil_div(n, (int64_t)kHistThreads * 4);
    hipLaunchKernelGGL(k_sort_hist<K>, dim3(hb < 256 ? hb : 256), dim3(kHistThreads), 0, st, keys, n, passes,
                       s.hist);
    bool swapped = false;
    for (int p = 0; p < passes; ++p, swapped = !swapped) {
        hipLaunchKernelGGL((k_sort_pass<K, kSortThreads>), dim3(tiles), dim3(kSortThreads), 0, st, swapped ? keys_tmp : keys,
                           swapped ? vals_tmp : vals, n, p, s.hist + p * kRadix, s.words, s.counters,
                           swapped ? keys : keys_tmp, swapped ? vals : vals_tmp);
        SPS_HIP(hipGetLastError());
    }
    return swapped;
}
template bool radix_sort_pairs<uint32_t>(uint32_t*, uint32_t*, uint32_t*, uint32_t*, int64_t, int, void*, hipStream_t);
template bool radix_sort_pairs<uint64_t>(uint64_t*, uint32_t*, uint64_t*, uint32_t*, int64_t, int, void*, hipStream_t);

template <typename K>
void launch_cand_keys(const CandD* c, int64_t n, int bits_t, int bits_w, K* keys, uint32_t* vals, void* scratch,
                      hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cand_keys<K>, dim3(grid1(n)), dim3(kThreads), 0, st, c, n, bits_t, bits_w, keys, vals,
                       static_cast<uint64_t*>(scratch), sort_clear(n));
    SPS_HIP(hipGetLastError());
}
template void launch_cand_keys<uint32_t>(const CandD*, int64_t, int, int, uint32_t*, uint32_t*, void*, hipStream_t);
template void launch_cand_keys<uint64_t>(const CandD*, int64_t, int, int, uint64_t*, uint32_t*, void*, hipStream_t);

template <typename K>
void launch_cand_from_keys(const K* keys, const uint32_t* vals, int64_t n, int bits_t, int bits_w, CandD* out,
                           hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cand_from_keys<K>, dim3(grid1(n)), dim3(kThreads), 0, st, keys, vals, n, bits_t, bits_w, out);
    SPS_HIP(hipGetLastError());
}
template void launch_cand_from_keys<uint32_t>(const uint32_t*, const uint32_t*, int64_t, int, int, CandD*, hipStream_t);
template void launch_cand_from_keys<uint64_t>(const uint64_t*, const uint32_t*, int64_t, int, int, CandD*, hipStream_t);

void launch_cand_ranges(const CandD* c, int64_t n, uint32_t* ranges, hipStream_t st) {
    if (n <= 0) return;
    const int64_t nb = ceil_div(n, (int64_t)kThreads * 8);
    hipLaunchKernelGGL(k_cand_ranges, dim3((uint32_t)(nb < 256 ? nb : 256)), dim3(kThreads), 0, st, c, n, ranges);
    SPS_HIP(hipGetLastError());
}

template <typename K>
void launch_cluster_keys(const CandD* c, const uint32_t* perm, const uint32_t* group, int64_t n, int member,
                         uint32_t base, int bits, K* keys, uint32_t* vals, void* scratch, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cluster_keys<K>, dim3(grid1(n)), dim3(kThreads), 0, st, c, perm, group, n, member, base, bits,
                       keys, vals, static_cast<uint64_t*>(scratch), sort_clear(n));
    SPS_HIP(hipGetLastError());
}
template void launch_cluster_keys<uint32_t>(const CandD*, const uint32_t*, const uint32_t*, int64_t, int, uint32_t, int,
                                            uint32_t*, uint32_t*, void*, hipStream_t);
template void launch_cluster_keys<uint64_t>(const CandD*, const uint32_t*, const uint32_t*, int64_t, int, uint32_t, int,
                                            uint64_t*, uint32_t*, void*, hipStream_t);

bool launch_cluster_small(const CandD* c, int64_t n, const int32_t* d_bins, uint32_t* perm, uint32_t* flags,
                          uint32_t* group, uint32_t* info, hipStream_t st) {
    if (n < 1 || n > 8 * kSmallThreads) return false;
    if (n <= kSmallThreads)
        hipLaunchKernelGGL(k_cluster_small<1>, dim3(1), dim3(kSmallThreads), 0, st, c, (int)n, d_bins, perm, flags,
                           group, info);
    else
        hipLaunchKernelGGL(k_cluster_small<8>, dim3(1), dim3(kSmallThreads), 0, st, c, (int)n, d_bins, perm, flags,
                           group, info);
    SPS_HIP(hipGetLastError());
    return true;
}

template <typename K>
void launch_cluster_groups(const K* keys, int64_t n, int bits, const int32_t* d_bins, int level, void* scratch,
                           uint32_t* flags, uint32_t* group, hipStream_t st) {
    if (n <= 0) return;
    const SortScratch s = sort_scratch(scratch, n);
    const int64_t tiles = ceil_div(n, (int64_t)kGroupTile);
    // (one fill from the counters to the last word)
    launch_fill_u64(static_cast<unsigned long long*>(scratch),
                    (int64_t)(s.words - static_cast<uint64_t*>(scratch)) + tiles, 0ull, st);
    hipLaunchKernelGGL(k_cluster_groups<K>, dim3((uint32_t)tiles), dim3(kThreads), 0, st, keys, n, bits, d_bins, level,
                       s.words, s.counters, flags, group);
    SPS_HIP(hipGetLastError());
}
template void launch_cluster_groups<uint32_t>(const uint32_t*, int64_t, int, const int32_t*, int, void*, uint32_t*,
                                              uint32_t*, hipStream_t);
template void launch_cluster_groups<uint64_t>(const uint64_t*, int64_t, int, const int32_t*, int, void*, uint32_t*,
                                              uint32_t*, hipStream_t);

void launch_cluster_delegates(const CandD* c, const uint32_t* perm, const uint32_t* gid, const uint32_t* flags,
                              int64_t n, unsigned long long* best, uint32_t* start, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_cluster_delegates, dim3((uint32_t)ceil_div(n, (int64_t)kDelItems * kWaves)), dim3(kThreads), 0,
                       st, c, perm, gid, flags, n, best, start);
    SPS_HIP(hipGetLastError());
}

void launch_delegate_keys(const CandD* c, const unsigned long long* best, int64_t ng, uint32_t base, uint32_t* keys,
                          uint32_t* vals, void* scratch, hipStream_t st) {
    if (ng <= 0) return;
    hipLaunchKernelGGL(k_delegate_keys, dim3(grid1(ng)), dim3(kThreads), 0, st, c, best, ng, base, keys, vals,
                       static_cast<uint64_t*>(scratch), sort_clear(ng));
    SPS_HIP(hipGetLastError());
}

void launch_delegate_out(const unsigned long long* best, const uint32_t* start, const uint32_t* order, int64_t ng,
                         int64_t n, int32_t* delegates, int64_t* sizes, hipStream_t st) {
    if (ng <= 0) return;
    hipLaunchKernelGGL(k_delegate_out, dim3(grid1(ng)), dim3(kThreads), 0, st, best, start, order, ng, n, delegates,
                       sizes);
    SPS_HIP(hipGetLastError());
}

void launch_pack_delegates(const CandD* c, const int32_t* del, const int64_t* size, int64_t ng, DelegateD* out,
                           hipStream_t st) {
    if (ng <= 0) return;
    hipLaunchKernelGGL(k_pack_delegates, dim3(grid1(ng)), dim3(kThreads), 0, st, c, del, size, ng, out);
    SPS_HIP(hipGetLastError());
}

void launch_fill_u64(unsigned long long* v, int64_t n, unsigned long long val, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_u64, dim3(grid1(n)), dim3(kThreads), 0, st, v, n, val);
    SPS_HIP(hipGetLastError());
}

void launch_select_delegates(const CandD* c, const int32_t* idx, int64_t nidx, const int32_t* begin, int64_t ngroups,
                             int32_t* out, hipStream_t st) {
    if (ngroups <= 0) return;
    if (ngroups > 0x7fffffffLL) throw Error(SPS_ERR_INVALID_ARGUMENT, "too many groups");
    hipLaunchKernelGGL(k_select_delegates, dim3((uint32_t)ngroups), dim3(64), 0, st, c, idx, nidx, begin, ngroups, out);
    SPS_HIP(hipGetLastError());
}

}  // namespace sps
