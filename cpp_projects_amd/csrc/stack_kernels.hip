// stack_kernels.hip -- stacked merge passes: up to six FDMT iterations (and,
// in the first pass, the init) per launch (tables: stack_plan.hpp).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "init_values.hpp"
#include "kernels.hpp"
#include "stack_plan.hpp"

namespace sps {

namespace {

constexpr int kWave = 64;
constexpr int kSegs = kStackTile / kWave;
constexpr int kTailSeg = kWave / kStackTailLanes;  // tail pieces a wave takes at a time

__device__ __forceinline__ float lds_at(const float* lds, int byte) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(lds) + byte);
}

// tree of 2^L leaves at byte offsets c[j] + u (left child first: the tail)
template <int L, int K = 1>
__device__ __forceinline__ float stack_tree(const float* lds, const int32_t (&c)[8], int u) {
    if constexpr (K >= (1 << L))
        return lds_at(lds, c[K - (1 << L)] + u);
    else
        return stack_tree<L, 2 * K>(lds, c, u) + stack_tree<L, 2 * K + 1>(lds, c, u);
}

// the lane's byte offsets of a row's leaves (u: 4 x the lane)
template <int L>
__device__ __forceinline__ void row_places(const StackRow& d, int u, int32_t (&c)[8]) {
#pragma unroll
    for (int j = 0; j < (1 << L); ++j) {
        if constexpr (L <= 2) c[j] = (int32_t)d.w[j] + u;
        else c[j] = (int32_t)((j % 2 ? d.w[j / 2] >> 16 : d.w[j / 2] & 0xffffu) << 2) + u;
    }
}

// times, row lengths and pitches are 32-bit (kStackMaxSamps)
struct StackArgs {
    uint32_t in_pitch, out_pitch;
    int plain_row0;  // row 0 is the sample itself (CFdmt), not 0 + the sample
    int la, lb;
    int ngroups;
    int tiles_per_block;
    int nsamps;
    int ntiles;
    int nrm_len;
};

// The rows of a stage over the block's waves, one row at a time; the next
// row's table entry is loaded meanwhile (kStackRowPad entries follow the last).
template <int WAVES, class F>
__device__ __forceinline__ void stage_rows(const StackRow* __restrict__ rows, int n, int wid, F&& row) {
    const StackRow* p = rows + wid;
    StackRow next = *p;
    for (int i = wid; i < n; i += WAVES) {  // wave-uniform
        const StackRow d = next;
        p += WAVES;
        next = *p;
        row(d);
    }
}

template <int L, int WAVES>
__device__ __forceinline__ void stage_a_rows(float* lds, const StackRow* __restrict__ rows, int n, int wid, int lane4) {
    stage_rows<WAVES>(rows, n, wid, [&](const StackRow& d) {
        int32_t c[8];
        row_places<L>(d, lane4, c);
        float v[kSegs];
#pragma unroll
        for (int s = 0; s < kSegs; ++s) v[s] = stack_tree<L>(lds, c, 4 * kWave * s);
        const int o = d.out + lane4;
#pragma unroll
        for (int s = 0; s < kSegs; ++s)
            *reinterpret_cast<float*>(reinterpret_cast<char*>(lds) + o + 4 * kWave * s) = v[s];
    });
}

// WHOLE: the tile ends inside the row.  EPI: 0 plain, 1 the S/N division by the
// kept channels' sqrtf (past the mask transform's extent), 2 by the mask
// transform's value of each sample where it has one.
template <int L, int EPI, bool WHOLE, int WAVES>
__device__ __forceinline__ void stage_b_rows(const float* lds, const StackArgs& a, const StackRow* __restrict__ rows,
                                             int n, float* __restrict__ out, const float* __restrict__ nrm, float dk,
                                             float rdk, int wid, int lane, int T) {
    float* __restrict__ const outT = out + T;
    if constexpr (EPI == 2) {
        // The mask transform's values of the next row are loaded before this
        // row's stores: a load after them would wait for them (8192 x 2^17,
        // where these are 6 % of the tiles: the pass took 2.56 ms, 2.34 so).
        constexpr int N = kSegs;
        auto divisors = [&](const StackRow& d, float (&v)[N]) {
            const float* nrow = nrm + (uint64_t)(uint32_t)d.out * (uint32_t)a.nrm_len;
#pragma unroll
            for (int s = 0; s < N; ++s) v[s] = nrow[min(T + lane + kWave * s, a.nrm_len - 1)];
        };
        float next[N];
        if (wid < n) divisors(rows[wid], next);
        for (int i = wid; i < n; i += WAVES) {  // wave-uniform
            const StackRow d = rows[i];
            float m[N];
#pragma unroll
            for (int s = 0; s < N; ++s) m[s] = next[s];
            if (i + WAVES < n) divisors(rows[i + WAVES], next);
            int32_t c[8];
            row_places<L>(d, 4 * lane, c);
            float* __restrict__ o = outT + (uint64_t)(uint32_t)d.out * a.out_pitch;
#pragma unroll
            for (int s = 0; s < N; ++s) {
                float v = stack_tree<L>(lds, c, 4 * kWave * s);
                const int t = T + lane + kWave * s;
                v = t < a.nrm_len ? v / sqrtf((float)((double)m[s] + 1.0E-8)) : div_rn(v, dk, rdk);
                if (WHOLE || t < a.nsamps) __builtin_nontemporal_store(v, &o[lane + kWave * s]);
            }
        }
        return;
    }
    stage_rows<WAVES>(rows, n, wid, [&](const StackRow& d) {
        constexpr int N = kSegs;
        int32_t c[8];
        row_places<L>(d, 4 * lane, c);
        float v[N];
#pragma unroll
        for (int s = 0; s < N; ++s) v[s] = stack_tree<L>(lds, c, 4 * kWave * s);
        if constexpr (EPI == 1) {
            // div_rn(v, dk, rdk): dk lies in [1e-4, 2^13] (sqrtf of up to 2^25
            // kept channels), so only the dividends need the range test, in one
            // rare branch
            bool slow = false;
            float q[N];
#pragma unroll
            for (int s = 0; s < N; ++s) {
                const float ax = fabsf(v[s]);
                slow = slow || !(ax >= 0x1p-60f && ax <= 0x1p60f);
                const float q0 = v[s] * rdk;
                q[s] = fmaf(fmaf(-q0, dk, v[s]), rdk, q0);
            }
            if (slow) {
#pragma unroll
                for (int s = 0; s < N; ++s) {
                    const float ax = fabsf(v[s]);
                    if (!(ax >= 0x1p-60f && ax <= 0x1p60f)) q[s] = v[s] / dk;
                }
            }
#pragma unroll
            for (int s = 0; s < N; ++s) v[s] = q[s];
        }
        // a wave-uniform row address and 32-bit lane offsets
        float* __restrict__ o = outT + (uint64_t)(uint32_t)d.out * a.out_pitch;
        if (WHOLE) {
#pragma unroll
            for (int s = 0; s < N; ++s) __builtin_nontemporal_store(v[s], &o[lane + kWave * s]);
        } else {
#pragma unroll
            for (int s = 0; s < N; ++s)
                if (T + lane + kWave * s < a.nsamps) o[lane + kWave * s] = v[s];
        }
    });
}

// KIND: 0 a state; 1 f32, 2 u8 waterfall, 3 ones (the pass builds state 0).
// The tables are separate __restrict__ arguments so that their wave-uniform
// reads are scalar loads: as members of a struct they may alias the output,
// every row then waited for the stores before it, and a second pass of the
// 4096 x 2^18 search took 5.0 ms.
template <int KIND, bool SNR, int THREADS>
__global__ void __launch_bounds__(THREADS, 8)
    k_stack(const StackArgs a, const void* __restrict__ in, float* __restrict__ out,
            const StackGroup* __restrict__ groups, const StackLeaf* __restrict__ leaves,
            const uint8_t* __restrict__ unit_leaf, const StackInitRow* __restrict__ inits,
            const StackRow* __restrict__ rows_a, const StackRow* __restrict__ rows_b,
            const StackTail* __restrict__ tails, const float* __restrict__ mu, const float* __restrict__ sigma,
            const uint8_t* __restrict__ keep, const float* __restrict__ nrm, const double* __restrict__ stats) {
    constexpr int kWaves = THREADS / kWave;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = (int)threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t logical = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t gi = logical % (uint32_t)a.ngroups;
    const uint32_t chunk = logical / (uint32_t)a.ngroups;
    const StackGroup g = groups[gi];
    const int k0 = (int)chunk * a.tiles_per_block;
    const int k1 = min(a.ntiles, k0 + a.tiles_per_block);
    if (k0 >= k1) return;  // block-uniform

    float dk = 1.0f, rdk = 1.0f;
    if (SNR) {
        // (in scalar registers: the 64 vector registers of 8 waves a SIMD are full)
        const float d = sqrtf((float)((double)(float)stats[4] + 1.0E-8));
        dk = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(d)));
        rdk = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(1.0f / d)));
    }
    // per slot: its unit's row in the input (for the init kinds a stack_slot
    // with the channel's place in chan[]), its time at T = 0 (the table
    // reads are unconditional, clamped to the group's units, so that all of
    // them are in flight together)
    uint32_t row_of[kStackSlots];
    int32_t tk[kStackSlots];
#pragma unroll
    for (int j = 0; j < kStackSlots; ++j)
        row_of[j] = unit_leaf[g.unit0 + min(tid + j * THREADS, g.nunits - 1)];
#pragma unroll
    for (int j = 0; j < kStackSlots; ++j) {
        const StackLeaf lf = leaves[g.leaf0 + row_of[j]];
        tk[j] = 4 * (min(tid + j * THREADS, g.nunits - 1) - lf.unit0) - lf.smax4;
        row_of[j] = KIND == 0 ? (uint32_t)lf.row : stack_slot((uint32_t)lf.row, row_of[j]);
    }
    // per channel {mu, sigma, 1/sigma, keep}
    __shared__ float4 chan[KIND == 0 ? 1 : kStackMaxChans];
    __shared__ int plain_all;
    if constexpr (KIND != 0) {
        if (tid == 0) plain_all = 1;
        __syncthreads();
        if (tid < g.nleaves) {
            float4 c = make_float4(0.0f, 1.0f, 1.0f, 1.0f);
            bool plain = KIND == 2;
            if (mu) {
                const int64_t ch = leaves[g.leaf0 + tid].row;
                if (keep[ch]) {
                    c.x = mu[ch];
                    c.y = sigma[ch];
                    c.z = 1.0f / c.y;
                    if (KIND == 2) plain = u8_init_plain(c.x, c.y);
                } else {
                    c.z = 0.0f;  // the fast quotient of v - 0 then is +0
                    c.w = 0.0f;
                }
            }
            if (!plain) plain_all = 0;
            chan[tid] = c;
        }
    }
    for (int i = tid; i < kStackTile; i += THREADS) lds[g.zero_off + i] = -0.0f;
    // the tails' tables, kept in LDS: a lane reads its own piece's
    StackTail* const tab = reinterpret_cast<StackTail*>(lds + g.tail_off);
    for (int i = tid; i < g.ntails * (int)(sizeof(StackTail) / 16); i += THREADS)
        reinterpret_cast<int4*>(tab)[i] = reinterpret_cast<const int4*>(tails + g.tail0)[i];

    // Every load is unconditional, at the row's edges with its time clamped
    // into the row (times outside are replaced at the commit): a register
    // that a load may or may not write is given its default first, and that
    // write waits for every load before it, one slot after the other.
    float4a buf[kStackSlots];
    uint32_t raw8[kStackSlots];
    // What follows from v is computed anew for every tile.  As loop invariants
    // the slots' rows, channels and LDS places spilled, and a reload from
    // scratch waits for every store before it: 2048 x 24576 f32 65 us, 39 so;
    // the S/N pass of 4096 x 2^18 3.10 and 2.87 ms.  The u8 kind's fit.
    auto anew = [](auto& v) {
        if constexpr (KIND != 2) asm volatile("" : "+v"(v));
    };
    const int row_end = KIND == 0 ? (int)a.in_pitch : a.nsamps;
    const int slot_f = wid * kWave;  // the wave's first unit of slot 0
    auto row_at = [&](int j) -> uint64_t {
        uint32_t r = row_of[j];
        anew(r);
        return (uint64_t)(KIND == 0 ? r : slot_chan(r)) * a.in_pitch;
    };
    auto load = [&](int j, uint64_t e) {
        if constexpr (KIND == 0) {
            buf[j] = *reinterpret_cast<const float4a*>(static_cast<const float*>(in) + e);
        } else if constexpr (KIND == 1) {
            const float4u w = *reinterpret_cast<const float4u*>(static_cast<const float*>(in) + e);
            buf[j] = float4a{w.x, w.y, w.z, w.w};
        } else if constexpr (KIND == 2) {
            raw8[j] = *reinterpret_cast<const u32u*>(static_cast<const uint8_t*>(in) + e);
        }
    };
    // every unit of the group lies inside the row
    auto inside = [&](int T) { return T >= g.smax4 && T + kStackTile + 4 <= row_end; };
    auto issue = [&](int T) {
        const bool in_row = inside(T);  // block-uniform
        if (!in_row && row_end < 4) return;
#pragma unroll
        for (int j = 0; j < kStackSlots; ++j) {
            if (slot_f + j * THREADS >= g.nunits) break;  // wave-uniform
            int t = T + tk[j];
            if (!in_row) t = max(0, min(row_end - 4, t));
            load(j, row_at(j) + (uint32_t)t);
        }
    };
    // KIND != 0: raw samples to row 0 of the channel
    auto row0 = [&](int j, float4a v) {
        uint32_t r = row_of[j];
        anew(r);
        const float4 c = chan[slot_place(r)];
        if (mu) {
            if (KIND == 2 && plain_all) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = v[e] - c.x;
                    const float q0 = x * c.z;
                    v[e] = fmaf(fmaf(-q0, c.y, x), c.z, q0);
                }
            } else {
                v = norm4(v, c.x, c.y, c.z);
                if (c.w == 0.0f) v = float4a{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        if (!a.plain_row0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = 0.0f + v[e];
        }
        return v;
    };
    auto raw = [&](int j) -> float4a {
        if constexpr (KIND == 3) return float4a{1.0f, 1.0f, 1.0f, 1.0f};
        else if constexpr (KIND == 2) return unpack_chunk<1>(raw8[j], buf[0]);
        else return buf[j];
    };
    auto commit = [&](int T) {
        const bool in_row = inside(T);  // block-uniform
        int u = tid;  // (one LDS address, the slots at constant offsets of it)
        anew(u);
        float* const mine = lds + 4 * u;
#pragma unroll
        for (int j = 0; j < kStackSlots; ++j) {
            if (slot_f + j * THREADS >= g.nunits) break;  // wave-uniform
            float4a v = raw(j);
            if (!in_row) {
                const int t = T + tk[j];
                if (KIND == 1 || KIND == 2) {
                    if (t >= 0 && t > row_end - 4) {  // cut by the row's end: sample by sample, 0 past it
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            v[e] = 0.0f;
                            if (t + e < row_end) {
                                const uint64_t x = row_at(j) + (uint32_t)(t + e);
                                if constexpr (KIND == 1) v[e] = static_cast<const float*>(in)[x];
                                else v[e] = (float)static_cast<const uint8_t*>(in)[x];
                            }
                        }
                    }
                }
                if constexpr (KIND != 0) v = row0(j, v);
                if (t < 0) v = float4a{-0.0f, -0.0f, -0.0f, -0.0f};
            } else {
                if constexpr (KIND != 0) v = row0(j, v);
            }
            if (u < g.nunits - j * THREADS) lds_store4(mine + 4 * j * THREADS, v);
        }
    };
    // init rows k >= 1 from the channels' row 0: v_0 = row 0, v_k = (v_{k-1} k
    // + row 0 (t - k)) / (k + 1), 0 for t < k
    auto init_rows = [&](int T) {
        for (int i = wid; i < g.ninit; i += kWaves) {  // wave-uniform
            const StackInitRow d = inits[g.init0 + i];
            for (int q0 = 0; q0 < d.n; q0 += kWave) {
                const int q = q0 + lane;
                if (q >= d.n) continue;
                float v = lds[d.c + q];
                for (int k = 1; k <= d.k; ++k) {
                    const float yk = (float)k + 1.0f;
                    v = div_rn(v * (float)k + lds[d.c + q - k], yk, 1.0f / yk);
                }
                const int t = T - d.t_off + q;
                if (t < d.k) v = t < 0 ? -0.0f : 0.0f;
                lds[d.out + q] = v;
            }
        }
    };
    auto stage_a = [&](auto ltag) {
        constexpr int L = decltype(ltag)::value;
        // the pieces of 8 lanes each, from the last wave down: the first
        // waves may have a row more
        for (int q = (kWaves - 1 - wid) * kTailSeg; q < g.ntails; q += kWaves * kTailSeg) {  // wave-uniform
            const int i = q + lane / kStackTailLanes, e = lane % kStackTailLanes;
            if (i < g.ntails && e < tab[i].n)
                *reinterpret_cast<float*>(reinterpret_cast<char*>(lds) + tab[i].out + 4 * e) =
                    stack_tree<L>(lds, tab[i].c, 4 * e);
        }
        stage_a_rows<L, kWaves>(lds, rows_a + g.row_a0, g.nrows_a, wid, 4 * lane);
    };
    auto stage_b = [&](int T) {
        const StackRow* rows = rows_b + g.row_b0;
        auto go = [&](auto ltag, auto etag, auto wtag) {
            stage_b_rows<decltype(ltag)::value, decltype(etag)::value, decltype(wtag)::value, kWaves>(
                lds, a, rows, g.nrows_b, out, nrm, dk, rdk, wid, lane, T);
        };
        auto depth = [&](auto etag, auto wtag) {
            if (a.lb == 3) go(std::integral_constant<int, 3>{}, etag, wtag);
            else if (a.lb == 2) go(std::integral_constant<int, 2>{}, etag, wtag);
            else if (a.lb == 1) go(std::integral_constant<int, 1>{}, etag, wtag);
            else go(std::integral_constant<int, 0>{}, etag, wtag);
        };
        const bool whole = T + kStackTile <= a.nsamps;
        if (SNR && (T < a.nrm_len || !whole)) depth(std::integral_constant<int, SNR ? 2 : 0>{}, std::false_type{});
        else if (whole) depth(std::integral_constant<int, SNR ? 1 : 0>{}, std::true_type{});
        else depth(std::integral_constant<int, 0>{}, std::false_type{});
    };

    // The next tile's units are committed between the stages (stage B no
    // longer reads the leaves), before stage B's stores: the wait for those
    // loads is a wait for every earlier memory operation of the wave, and
    // the stores before it are by then a stage old.
    if constexpr (KIND != 0) __syncthreads();  // the channel table, which issue and commit read
    issue(k0 * kStackTile);
    for (int k = k0 - 1; k < k1; ++k) {  // k0 - 1: the first commit alone
        const int T = k * kStackTile;
        if (k >= k0) {  // block-uniform, as are the branches below
            if (a.la == 3) stage_a(std::integral_constant<int, 3>{});
            else if (a.la == 2) stage_a(std::integral_constant<int, 2>{});
            else stage_a(std::integral_constant<int, 1>{});
            __syncthreads();
        }
        if (k + 1 < k1) commit(T + kStackTile);
        if (k + 2 < k1) issue(T + 2 * kStackTile);
        if (k >= k0) stage_b(T);
        __syncthreads();  // the next leaves are there, stage B is done
        if constexpr (KIND != 0) {
            if (g.ninit && k + 1 < k1) {
                init_rows(T + kStackTile);
                __syncthreads();
            }
        }
    }
}

// Consecutive tiles a block takes.  512 blocks run at a time (two a CU), and a
// block's setup costs almost half a tile: up to three tiles a block as soon as
// the tiles are more than 512 (2048 x 24576, 3072 tiles: 75 us at one, 65 at
// three, 63 at six; 1024 x 20000, 1413 tiles: 33 and 27.5 at three), more from
// 2048 blocks on (6256 tiles: 99 us at three, 104 at four, 126 at twelve, whose
// last blocks run alone).  More than 32 tiles a block reach too far apart in
// time for the groups to share L2 (4096 x 2^18: 5.4 ms at 32, 5.9 at 128).
int tiles_per_block(int64_t tiles) {
    const int64_t few = std::min<int64_t>(3, ceil_div(tiles, 512));
    return (int)std::max(few, std::min<int64_t>(32, tiles / 2048));
}

template <int KIND>
void stack_launch(const StackPassDev& p, const StackArgs& a, const void* in, const ChanNorm& n, float* out,
                  const MergeEpilogue* snr, uint32_t nb, hipStream_t st) {
    const size_t lds = sizeof(float) * (size_t)p.lds_floats;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(p.threads), lds, st, a, in, out,
                           static_cast<const StackGroup*>(p.groups), static_cast<const StackLeaf*>(p.leaves),
                           p.unit_leaf, static_cast<const StackInitRow*>(p.inits),
                           static_cast<const StackRow*>(p.rows_a), static_cast<const StackRow*>(p.rows_b),
                           static_cast<const StackTail*>(p.tails), n.mu, n.sigma, n.keep, snr ? snr->nrm : nullptr,
                           snr ? snr->stats : nullptr);
    };
    if (p.threads == kStackFew4) snr ? go(&k_stack<KIND, true, kStackFew4>) : go(&k_stack<KIND, false, kStackFew4>);
    else if (p.threads == kStackFew16) snr ? go(&k_stack<KIND, true, kStackFew16>) : go(&k_stack<KIND, false, kStackFew16>);
    else snr ? go(&k_stack<KIND, true, kStackThreads>) : go(&k_stack<KIND, false, kStackThreads>);
}

template <int KIND, bool SNR>
void stack_attribute() {
    SPS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_stack<KIND, SNR, kStackThreads>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(float) * kStackLdsFloats)));
}

}  // namespace

// once per device: the attribute belongs to the function on it
void prepare_stack_kernels() {
    static std::mutex m;
    static uint64_t done = 0;
    int dev = 0;
    SPS_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(m);
    if (dev < 64 && (done >> dev & 1)) return;
    stack_attribute<0, false>();
    stack_attribute<0, true>();
    stack_attribute<1, false>();
    stack_attribute<1, true>();
    stack_attribute<2, false>();
    stack_attribute<2, true>();
    stack_attribute<3, false>();
    stack_attribute<3, true>();
    if (dev < 64) done |= (uint64_t)1 << dev;
}

void launch_stack_pass(const StackPassDev& p, int kind, const void* in, int64_t in_pitch, const ChanNorm* norm,
                       bool plain_row0, float* out, int64_t out_pitch, int64_t nsamps, hipStream_t st,
                       const MergeEpilogue* snr) {
    if (p.ngroups <= 0 || nsamps <= 0) return;
    if (kind == 0 && (in_pitch % 4 != 0 || reinterpret_cast<uintptr_t>(in) % 16 != 0))
        throw Error(SPS_ERR_INVALID_ARGUMENT, "stacked pass needs a 16-byte aligned input state");
    if ((kind != 0) != p.init) throw Error(SPS_ERR_INVALID_ARGUMENT, "stacked pass tables do not match its input");
    if (p.lds_floats <= 0 || p.lds_floats > kStackLdsFloats)
        throw Error(SPS_ERR_INVALID_ARGUMENT, "stacked pass LDS out of range");
    if (p.threads != kStackThreads && p.threads != kStackFew16 && p.threads != kStackFew4)
        throw Error(SPS_ERR_INVALID_ARGUMENT, "stacked pass block size");
    StackArgs a{};
    if (nsamps > kStackMaxSamps || in_pitch > kStackMaxSamps + 4 || out_pitch > kStackMaxSamps + 4)
        throw Error(SPS_ERR_INVALID_ARGUMENT, "rows too long for a stacked pass");
    a.in_pitch = (uint32_t)in_pitch;
    a.plain_row0 = plain_row0 ? 1 : 0;
    a.out_pitch = (uint32_t)out_pitch;
    a.ngroups = (int)p.ngroups;
    a.la = p.la;
    a.lb = p.lb;
    a.nsamps = (int)nsamps;
    a.ntiles = (int)ceil_div(nsamps, (int64_t)kStackTile);
    a.nrm_len = snr ? (int)snr->nrm_len : 0;
    ChanNorm n{};
    if (norm) n = *norm;
    a.tiles_per_block = tiles_per_block(p.ngroups * a.ntiles);
    const int64_t nb = p.ngroups * ceil_div((int64_t)a.ntiles, (int64_t)a.tiles_per_block);
    if (nb > 0x7fffffffLL) throw Error(SPS_ERR_INVALID_ARGUMENT, "merge grid too large");
    switch (kind) {
        case 0: stack_launch<0>(p, a, in, n, out, snr, (uint32_t)nb, st); break;
        case 1: stack_launch<1>(p, a, in, n, out, snr, (uint32_t)nb, st); break;
        case 2: stack_launch<2>(p, a, in, n, out, snr, (uint32_t)nb, st); break;
        case 3: stack_launch<3>(p, a, in, n, out, snr, (uint32_t)nb, st); break;
        default: throw Error(SPS_ERR_INVALID_ARGUMENT, "unknown stacked pass input");
    }
    SPS_HIP(hipGetLastError());
}

}  // namespace sps
