// api.cpp -- the extern "C" boundary of libsps (declared in include/sps.h).
// Every entry point converts C++ exceptions into an sps_status and records
// the message for sps_last_error().
#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "abi.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "scratch.hpp"
#include "plan.hpp"
#include "stack_plan.hpp"

using namespace sps;

namespace sps {
thread_local std::string g_last_error;
}

namespace {

template <class T>
void upload(DevBuf& b, const std::vector<T>& v, hipStream_t st) {
    b.ensure(std::max<size_t>(sizeof(T) * v.size(), 16));
    if (!v.empty()) SPS_HIP(hipMemcpyAsync(b.p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice, st));
}

int bitlen(uint64_t v) {
    int b = 0;
    while (v) {
        ++b;
        v >>= 1;
    }
    return b;
}

int64_t round_up(int64_t a, int64_t m) { return ((a + m - 1) / m) * m; }

}  // namespace

// ---------------------------------------------------------------------------
// FDMT handle
// ---------------------------------------------------------------------------
struct sps_fdmt {
    std::unique_ptr<FdmtPlan> plan;    // plan-based FDMT
    std::unique_ptr<CFdmtPlan> cplan;  // legacy CFdmt
    EnginePlan eng;
    int64_t pitch = 0;                 // internal state pitch (floats)
    bool uploaded = false;
    DevBuf d_grid, d_grid_off, d_chan_row_off;
    std::vector<std::unique_ptr<DevBuf>> d_rows;  // per iteration: RowDescD of its live output rows (run_single)
    std::vector<int64_t> d_rows_n;                // per iteration: number of those rows
    DevBuf state_a, state_b;
    int64_t rows_a = 0, rows_b = 0;    // capacity of the ping-pong states in rows
    DevBuf host_in, host_out;          // device copies for the host-pointer calls
    int dmax = 0;                      // largest init dt of any channel
    int grid_consec = 0;               // every channel's init dts are 0, 1, ..., K-1 with K <= 5
    bool init_in_pass = false;         // the first stacked pass may build state 0 (dts 0, 1, ..., K-1 with K <= 16)
    // adjoint: launches from the last iteration down (depth iterations each),
    // their tables, and states of its own, so that execute's stay where a
    // caller's captured graph has them.  Where those do not fit beside execute's
    // and no graph has taken execute's, both use the same (adj_shared).
    struct AdjPass {
        int depth = 0;
        int64_t prev_rows = 0;
        DevBuf off, users;
    };
    bool adj_built = false;
    std::vector<std::unique_ptr<AdjPass>> adj;
    DevBuf adj_a, adj_b;
    bool adj_shared = false;
    bool states_captured = false;  // an execute was captured: its states stay where they are

    // Pass schedule as callers set and read it: iterations per entry (1..3, or
    // 1..4 with a staging mode), summing to niters.  The launches are the
    // stacked passes below, split by the iteration count alone; the schedule
    // is what stage times and bytes are reported by.
    std::vector<int> schedule;
    int staging = 0;          // as set (set_staged)
    bool staged = false;      // ... and not 0
    bool ran_fused0 = false;  // the last execution's first pass built state 0 itself (stage accounting)

    // A launch of the stacked kernel: `depth` iterations from i0 on
    // (stack_plan.hpp); the first builds state 0 itself when `init`.
    struct StackPass {
        int i0 = 1, depth = 0;
        StackPassDev dev;
    };
    std::vector<StackPass> passes;
    DevBuf pass_tables;  // every pass's tables
    DevBuf in_copy;      // the waterfall, where the image overwrites it (copy_overlapped)
    bool passes_ready = false;
    bool weigh_init = true;  // the first pass may leave state 0 to the separate init where that is faster

    void init_layout() {
        pitch = round_up(eng.nsamps, 4);
        dmax = eng.max_init_dt();
        int64_t kmax = 0;
        bool consec = true;
        for (int64_t c = 0; c < eng.nchans && consec; ++c) {
            const int64_t g0 = eng.grid_off[(size_t)c], K = eng.grid_off[(size_t)c + 1] - g0;
            consec = K >= 1;
            kmax = std::max(kmax, K);
            for (int64_t k = 0; k < K && consec; ++k) consec = eng.grid[(size_t)(g0 + k)] == k;
        }
        grid_consec = consec && kmax <= 5;
        init_in_pass = consec && kmax <= 16 && eng.init_mode != kInitRestrict;
        // state 0 in A; pass outputs alternate B, A, B, ... and rows only
        // shrink with the iteration, so A needs rows[0] and B rows[1]
        rows_a = eng.rows[0];
        rows_b = eng.niters >= 1 ? eng.rows[1] : 0;
        for (int i = 1; i <= eng.niters; ++i) {
            SPS_REQUIRE((int64_t)eng.iter[(size_t)i].size() == eng.rows[(size_t)i], "plan rows do not cover the state");
            for (int64_t r = 0; r < eng.rows[(size_t)i]; ++r)
                SPS_REQUIRE(eng.iter[(size_t)i][(size_t)r].out_row == r, "plan rows out of order");
            rows_a = std::max(rows_a, eng.rows[(size_t)i]);
        }
        compute_live();
        set_schedule(default_schedule(eng.niters));
    }

    // Rows of an intermediate state that no delivered output row depends on
    // (the plan's dt grid per sub-band is wider than what the last merges
    // read) are never computed: skipping them changes no output value.
    std::vector<std::vector<uint8_t>> live;  // per state
    DevBuf d_live0;                          // state-0 flags for the init kernels
    void compute_live() {
        const int n = eng.niters;
        live.assign((size_t)n + 1, {});
        for (int i = 0; i <= n; ++i) live[(size_t)i].assign((size_t)eng.rows[(size_t)i], 0);
        for (int64_t r = 0; r < eng.rows[(size_t)n]; ++r) live[(size_t)n][(size_t)r] = r < eng.out_rows ? 1 : 0;
        for (int i = n; i >= 1; --i)
            for (const auto& rd : eng.iter[(size_t)i]) {
                if (!live[(size_t)i][(size_t)rd.out_row]) continue;
                live[(size_t)i - 1][(size_t)rd.tail_row] = 1;
                if (rd.head_row >= 0) live[(size_t)i - 1][(size_t)rd.head_row] = 1;
            }
    }
    int64_t live_rows(int i) const {
        int64_t c = 0;
        for (auto v : live[(size_t)i]) c += v;
        return c;
    }

    static constexpr int kMaxDepth = 3, kMaxStagedDepth = 4;  // iterations of a schedule entry
    static std::vector<int> default_schedule(int n) {
        std::vector<int> s;
        while (n > 0) {
            const int d = (n % kMaxDepth == 1 && n > kMaxDepth) ? 2 : std::min(n, kMaxDepth);
            s.push_back(d);
            n -= d;
        }
        return s;
    }

    void set_schedule(const std::vector<int>& s) {
        int sum = 0;
        const int maxd = staged ? kMaxStagedDepth : kMaxDepth;
        for (int d : s) {
            SPS_REQUIRE(d >= 1 && d <= maxd, staged ? "staged fusion depth must be 1..4" : "fusion depth must be 1..3");
            sum += d;
        }
        SPS_REQUIRE(sum == eng.niters, "schedule must cover every iteration");
        schedule = s;
    }

    static void set_group_shape(int floats, int rows, int tiles) {
        SPS_REQUIRE(floats >= 2048 && floats <= 9216, "group window must be 2048..9216 floats");
        SPS_REQUIRE(rows >= 1 && rows <= 64, "group rows must be 1..64");
        SPS_REQUIRE(tiles >= 1 && tiles <= 512, "tiles per block must be 1..512");
    }

    // mode 0 limits schedule entries to 3 iterations, modes 1..4 to 4
    void set_staged(int mode) {
        SPS_REQUIRE(mode >= 0 && mode <= 4, "staging mode must be 0..4");
        staging = mode;
        staged = mode > 0;
        for (int d : schedule)
            if (d > (staged ? kMaxStagedDepth : kMaxDepth)) {
                schedule = default_schedule(eng.niters);
                break;
            }
    }

    // The launches: as few passes as kStackMaxDepth iterations each allow, the
    // iterations split evenly, the deeper passes first (the first reads the
    // waterfall rather than a state).  Both passes of 4096 x 2^18 (12
    // iterations): 6 + 6 5.13-5.26 ms, 4 + 4 + 4 5.31, 5 + 4 + 3 5.5; shorter rows
    // gain a launch.
    std::vector<int> pass_depths() const {
        std::vector<int> d;
        if (eng.nsamps > kStackMaxSamps) {
            d.assign((size_t)eng.niters, 1);
            return d;
        }
        const int np = (eng.niters + kStackMaxDepth - 1) / kStackMaxDepth;
        for (int k = 0, left = eng.niters; k < np; ++k, left -= d.back()) d.push_back((left + np - k - 1) / (np - k));
        return d;
    }
    void ensure_passes(hipStream_t st) {
        if (passes_ready || eng.niters == 0 || eng.nsamps > kStackMaxSamps) return;
        passes.clear();
        prepare_stack_kernels();
        std::vector<uint8_t> host;  // one upload for all of them
        auto put = [&](const auto& v) -> size_t {
            const size_t at = (host.size() + 255) / 256 * 256;
            host.resize(at + sizeof(v[0]) * v.size());
            if (!v.empty()) std::memcpy(host.data() + at, v.data(), sizeof(v[0]) * v.size());
            return at;
        };
        struct At {
            size_t groups, leaves, unit_leaf, inits, rows_a, rows_b, tails;
        };
        std::vector<At> at;
        int i0 = 1;
        for (int depth : pass_depths()) {
            bool init = i0 == 1 && init_in_pass;
            StackTables t;
            if (init) {
                // a first pass whose trees need more init rows than one LDS
                // window holds, or so many that they cost more than a state 0
                // in memory, keeps the separate init
                try {
                    // (the separate init's grid takes 65535 channels)
                    t = build_stack_pass(eng, live, i0, depth, true, weigh_init && eng.nchans <= 65535);
                    init = t.init;
                } catch (const std::runtime_error&) {
                    init = false;
                }
            }
            if (!init) t = build_stack_pass(eng, live, i0, depth, false);
            at.push_back(At{put(t.groups), put(t.leaves), put(t.unit_leaf), put(t.inits), put(t.rows_a), put(t.rows_b),
                            put(t.tails)});
            StackPass ps;
            ps.i0 = i0;
            ps.depth = depth;
            ps.dev.ngroups = (int64_t)t.groups.size();
            ps.dev.la = t.la;
            ps.dev.lb = t.lb;
            ps.dev.lds_floats = t.lds_floats;
            ps.dev.init = t.init;
            ps.dev.threads = stack_threads(t);
            passes.push_back(ps);
            i0 += depth;
        }
        upload(pass_tables, host, st);
        for (size_t k = 0; k < passes.size(); ++k) {
            const uint8_t* base = pass_tables.as<uint8_t>();
            StackPassDev& d = passes[k].dev;
            d.groups = base + at[k].groups;
            d.leaves = base + at[k].leaves;
            d.unit_leaf = base + at[k].unit_leaf;
            d.inits = base + at[k].inits;
            d.rows_a = base + at[k].rows_a;
            d.rows_b = base + at[k].rows_b;
            d.tails = base + at[k].tails;
        }
        SPS_HIP(hipStreamSynchronize(st));  // the host copy ends with this call
        passes_ready = true;
    }

    void ensure_device(hipStream_t st) {
        if (uploaded) return;
        upload(d_grid, eng.grid, st);
        upload(d_grid_off, eng.grid_off, st);
        upload(d_chan_row_off, eng.chan_row_off, st);
        if (eng.nsamps > kStackMaxSamps) {
            d_rows.clear();
            d_rows_n.clear();
            for (int i = 0; i <= eng.niters; ++i) {
                d_rows.emplace_back(new DevBuf());
                std::vector<RowDescD> rd;
                for (const auto& r : eng.iter[(size_t)i])
                    if (live[(size_t)i][(size_t)r.out_row]) rd.push_back({r.out_row, r.tail_row, r.head_row, r.offset});
                upload(*d_rows.back(), rd, st);
                d_rows_n.push_back((int64_t)rd.size());
            }
        }
        upload(d_live0, live[0], st);
        SPS_HIP(hipStreamSynchronize(st));
        uploaded = true;
    }

    // The separate init's grid takes 65535 channels.  Larger plans run where a
    // first pass that builds state 0 itself was asked for (staging mode 2 or 4,
    // more than one schedule entry) and are refused otherwise.
    void check_channels(bool ones) const {
        const bool asked = (staging == 2 || staging == 4) && schedule.size() >= 2 && grid_consec &&
                           eng.init_mode == kInitMean && !ones;
        if (eng.nchans > 65535 && !asked) throw Error(SPS_ERR_INVALID_ARGUMENT, "more than 65535 channels");
    }

    // What execute needs on the device before its launches: the passes'
    // tables, those of the separate init or merges where they run, and the
    // states.
    void prepare(hipStream_t st) {
        ensure_passes(st);
        if (passes.empty() || !passes[0].dev.init) ensure_device(st);
    }
    // Rows of the two states that execute's passes write: state 0 (unless the
    // first pass builds it) and the outputs of passes 1, 3, ... in A, of
    // passes 0, 2, ... in B; the last pass writes the caller's image.
    void state_rows(int64_t& a, int64_t& b) const {
        a = rows_a;
        b = rows_b;
        if (eng.niters > 0 && passes.empty()) return;  // one merge per launch
        a = !passes.empty() && passes[0].dev.init ? 0 : eng.rows[0];
        b = 0;
        for (size_t k = 0; k + 1 < passes.size(); ++k) {
            const int64_t r = eng.rows[(size_t)(passes[k].i0 + passes[k].depth - 1)];
            (k % 2 ? a : b) = std::max(k % 2 ? a : b, r);
        }
        if (eng.niters == 0) a = b = 0;
    }
    void ensure_states(hipStream_t st) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cap) != hipSuccess) (void)hipGetLastError();
        if (cap != hipStreamCaptureStatusNone) states_captured = true;
        auto states = [&] {
            int64_t a, b;
            state_rows(a, b);
            if (a) state_a.ensure(sizeof(float) * (size_t)checked_mul(a, pitch, "state"));
            if (b) state_b.ensure(sizeof(float) * (size_t)checked_mul(b, pitch, "state"));
        };
        try {
            states();
        } catch (const Error& e) {
            // a state 0 that the first pass gave away and that does not fit
            if (e.status != SPS_ERR_NO_MEMORY || !weigh_init || !init_in_pass || passes.empty() || passes[0].dev.init)
                throw;
            weigh_init = false;
            passes_ready = false;
            ensure_passes(st);
            states();
        }
    }

    // A plan of one pass that builds state 0 reads the waterfall while other
    // blocks write the image.  Where the two overlap it runs from a copy of the
    // waterfall; every other plan has written a state before the image.
    // overlap_bytes: the size of that copy, 0 where none is needed.
    size_t overlap_bytes(const void* in, int in_u8, int64_t in_pitch, int64_t nsamps, const float* out,
                         int64_t out_pitch) const {
        if (passes.size() != 1 || !passes[0].dev.init || !in) return 0;
        const size_t ib = (size_t)((eng.nchans - 1) * in_pitch + nsamps) * (in_u8 ? 1 : sizeof(float));
        const size_t ob = (size_t)((eng.out_rows - 1) * out_pitch + nsamps) * sizeof(float);
        const uintptr_t i = reinterpret_cast<uintptr_t>(in), o = reinterpret_cast<uintptr_t>(out);
        return i < o + ob && o < i + ib ? ib : 0;
    }
    const void* copy_overlapped(const void* in, size_t bytes, hipStream_t st) {
        in_copy.ensure(bytes);
        SPS_HIP(hipMemcpyAsync(in_copy.p, in, bytes, hipMemcpyDeviceToDevice, st));
        return in_copy.p;
    }

    // Runs init + merges over nsamps samples (nsamps <= eng.nsamps) writing the
    // final rows to out (pitch out_pitch).  sa/sb: ping-pong states with pitch p.
    // ev (optional): one event recorded after the init and after every merge.
    // snr (optional): S/N epilogue fused into the last merge; aux: mask transform.
    void run(const void* in, int in_u8, int ones, int64_t in_pitch, const ChanNorm* norm, int64_t nsamps, float* out,
             int64_t out_pitch, float* sa, float* sb, int64_t p, hipStream_t st, hipEvent_t* ev = nullptr,
             const MergeEpilogue* snr = nullptr, bool aux = false) {
        SPS_REQUIRE(!snr || eng.niters > 0, "the S/N epilogue needs at least one merge");
        const ChanNorm* nm = norm;
        if (!aux) ran_fused0 = false;
        if (eng.niters == 0) {
            launch_fdmt_init(eng.init_mode, in, in_u8, ones, in_pitch, nm, eng.nchans, nsamps, d_grid.as<int32_t>(),
                             d_grid_off.as<int64_t>(), d_chan_row_off.as<int64_t>(), out, out_pitch, st, dmax,
                             nullptr, grid_consec);
            if (ev) SPS_HIP(hipEventRecord(ev[0], st));
            return;
        }
        check_channels(ones != 0);
        if (eng.nsamps > kStackMaxSamps) {
            run_single(in, in_u8, ones, in_pitch, nm, nsamps, out, out_pitch, sa, sb, p, st, ev, snr);
            return;
        }
        ensure_passes(st);
        const bool fused0 = passes[0].dev.init;
        if (!aux) ran_fused0 = fused0;
        if (!ones)
            if (const size_t n = overlap_bytes(in, in_u8, in_pitch, nsamps, out, out_pitch))
                in = copy_overlapped(in, n, st);
        if (!fused0)
            launch_fdmt_init(eng.init_mode, in, in_u8, ones, in_pitch, nm, eng.nchans, nsamps, d_grid.as<int32_t>(),
                             d_grid_off.as<int64_t>(), d_chan_row_off.as<int64_t>(), sa, p, st, dmax,
                             d_live0.as<uint8_t>(), grid_consec);
        if (ev) SPS_HIP(hipEventRecord(ev[0], st));
        size_t done = 0;  // schedule entries whose event is recorded
        int entry_end = 0;
        for (size_t k = 0; k < passes.size(); ++k) {
            const StackPass& ps = passes[k];
            const int top = ps.i0 + ps.depth - 1;
            const float* src = (k % 2 == 0) ? sa : sb;
            const bool last = (top == eng.niters);
            float* dst = last ? out : ((k % 2 == 0) ? sb : sa);
            const bool first = k == 0 && fused0;
            const int kind = !first ? 0 : ones ? 3 : in_u8 ? 2 : 1;
            launch_stack_pass(ps.dev, kind, first ? in : src, first ? in_pitch : p, first ? nm : nullptr,
                              eng.init_mode == kInitCFdmt, dst, last ? out_pitch : p, nsamps, st, last ? snr : nullptr);
            // a joined schedule entry ends with its launch
            while (ev && done < schedule.size() && entry_end + schedule[done] <= top) {
                entry_end += schedule[done++];
                SPS_HIP(hipEventRecord(ev[done], st));
            }
        }
    }

    // Rows beyond the stacked kernel's 32-bit times: the init and one launch
    // per iteration.
    void run_single(const void* in, int in_u8, int ones, int64_t in_pitch, const ChanNorm* nm, int64_t nsamps,
                    float* out, int64_t out_pitch, float* sa, float* sb, int64_t p, hipStream_t st, hipEvent_t* ev,
                    const MergeEpilogue* snr) {
        launch_fdmt_init(eng.init_mode, in, in_u8, ones, in_pitch, nm, eng.nchans, nsamps, d_grid.as<int32_t>(),
                         d_grid_off.as<int64_t>(), d_chan_row_off.as<int64_t>(), sa, p, st, dmax,
                         d_live0.as<uint8_t>(), grid_consec);
        if (ev) SPS_HIP(hipEventRecord(ev[0], st));
        size_t done = 0;
        int entry_end = 0;
        for (int i = 1; i <= eng.niters; ++i) {
            const float* src = (i - 1) % 2 == 0 ? sa : sb;
            const bool last = i == eng.niters;
            float* dst = last ? out : (i % 2 == 0 ? sa : sb);
            launch_fdmt_merge(src, p, dst, last ? out_pitch : p, d_rows[(size_t)i]->as<RowDescD>(),
                              d_rows_n[(size_t)i], nsamps, last ? eng.out_rows : INT64_MAX, st, last ? snr : nullptr);
            while (ev && done < schedule.size() && entry_end + schedule[done] <= i) {
                entry_end += schedule[done++];
                SPS_HIP(hipEventRecord(ev[done], st));
            }
        }
    }

    void build_adjoint(hipStream_t st) {
        if (adj_built) return;
        adj.clear();
        std::vector<std::vector<std::vector<std::pair<int64_t, int64_t>>>> users((size_t)eng.niters + 1);
        for (int i = 1; i <= eng.niters; ++i) {
            auto& us = users[(size_t)i];
            us.resize((size_t)eng.rows[(size_t)i - 1]);
            for (const auto& r : eng.iter[(size_t)i]) {
                us[(size_t)r.tail_row].push_back({r.out_row, 0});
                if (r.head_row >= 0) us[(size_t)r.head_row].push_back({r.out_row, r.offset});
            }
            for (auto& u : us) std::sort(u.begin(), u.end());
        }
        int64_t need[2] = {0, 0};
        const std::vector<int> depths = adjoint_depths(eng);
        for (size_t k = 0, top = (size_t)eng.niters; k < depths.size(); ++k) {
            const int depth = depths[k];
            const int low = (int)top - depth + 1;
            std::unique_ptr<AdjPass> pass(new AdjPass());
            pass->depth = depth;
            pass->prev_rows = eng.rows[(size_t)low - 1];
            std::vector<int64_t> off(1, 0);
            std::vector<AdjUser> tab;
            // users of row at iteration i, depth first; an empty sum in
            // between adds nothing
            std::function<void(int64_t, int, int64_t)> walk = [&](int64_t row, int i, int64_t shift) {
                for (const auto& u : users[(size_t)i][(size_t)row]) {
                    const size_t before = tab.size();
                    if (i == (int)top) {
                        tab.push_back({shift + u.second, (uint32_t)u.first, 0});
                    } else {
                        walk(u.first, i + 1, shift + u.second);
                        if (tab.size() > before) ++tab.back().closes;
                    }
                }
            };
            for (int64_t p = 0; p < pass->prev_rows; ++p) {
                walk(p, low, 0);
                off.push_back((int64_t)tab.size());
            }
            upload(pass->off, off, st);
            upload(pass->users, tab, st);
            SPS_HIP(hipStreamSynchronize(st));
            need[k % 2] = std::max(need[k % 2], pass->prev_rows);
            adj.push_back(std::move(pass));
            top = (size_t)low - 1;
        }
        auto bytes = [&](int64_t rows) { return sizeof(float) * (size_t)checked_mul(rows, pitch, "state"); };
        try {
            adj_a.ensure(bytes(std::max<int64_t>(need[0], 1)));
            if (need[1]) adj_b.ensure(bytes(need[1]));
        } catch (const Error& e) {
            if (e.status != SPS_ERR_NO_MEMORY || states_captured) throw;
            adj_a.release();
            adj_b.release();
            prepare(st);
            int64_t a, b;
            state_rows(a, b);
            state_a.release();  // (waits for what still uses them)
            state_b.release();
            state_a.ensure(bytes(std::max<int64_t>(std::max(a, need[0]), 1)));
            state_b.ensure(bytes(std::max<int64_t>(std::max(b, need[1]), 1)));
            adj_shared = true;
        }
        adj_built = true;
    }
};

static void finish_create(sps_fdmt* h) {
    h->init_layout();
}

extern "C" {

SPS_API const char* sps_last_error(void) { return g_last_error.c_str(); }
SPS_API int sps_version(void) { return 100; }

SPS_API sps_status sps_device_count(int* h_count) {
    return guarded([&] {
        SPS_REQUIRE(h_count, "null output");
        int n = 0;
        hipError_t e = hipGetDeviceCount(&n);
        *h_count = (e == hipSuccess) ? n : 0;
    });
}

SPS_API sps_status sps_release_scratch(void) {
    return guarded([&] { scratch_trim(); });
}

SPS_API sps_status sps_fdmt_create(float f_min, float f_max, int64_t nchans, int64_t nsamps, float tsamp,
                                   int64_t dt_max, int64_t dt_step, int64_t dt_min, int init_mode, sps_fdmt** out) {
    return guarded([&] {
        SPS_REQUIRE(out, "null output handle");
        *out = nullptr;
        std::unique_ptr<sps_fdmt> h(new sps_fdmt());
        h->plan.reset(new FdmtPlan(f_min, f_max, nchans, nsamps, tsamp, dt_max, dt_step, dt_min));
        h->eng = h->plan->lower(init_mode);
        finish_create(h.get());
        *out = h.release();
    });
}

SPS_API sps_status sps_cfdmt_create(float f_min, float f_max, int nchan, int cols, int imaxdt, sps_fdmt** out) {
    return guarded([&] {
        SPS_REQUIRE(out, "null output handle");
        *out = nullptr;
        std::unique_ptr<sps_fdmt> h(new sps_fdmt());
        h->cplan.reset(new CFdmtPlan(f_min, f_max, nchan, cols, imaxdt));
        h->eng = h->cplan->lower();
        finish_create(h.get());
        *out = h.release();
    });
}

SPS_API sps_status sps_fdmt_destroy(sps_fdmt* h) {
    return guarded([&] {
        delete h;
        scratch_trim();
    });
}

SPS_API sps_status sps_fdmt_get_niters(const sps_fdmt* h, int64_t* n) {
    return guarded([&] {
        SPS_REQUIRE(h && n, "null argument");
        *n = h->eng.niters;
    });
}

SPS_API sps_status sps_fdmt_get_state_shape(const sps_fdmt* h, int64_t iter, int64_t* s5) {
    return guarded([&] {
        SPS_REQUIRE(h && s5, "null argument");
        SPS_REQUIRE(iter >= 0 && iter <= h->eng.niters, "iteration out of range");
        if (h->plan) {
            h->plan->state_shape(iter, s5);
        } else {
            const auto& c = *h->cplan;
            const int q = c.quant[(size_t)iter];
            int mn = INT32_MAX, mx = 0;
            for (int i = 0; i < q; ++i) {
                int r = c.cumsum[(size_t)iter][(size_t)i + 1] - c.cumsum[(size_t)iter][(size_t)i];
                mn = std::min(mn, r);
                mx = std::max(mx, r);
            }
            s5[0] = q;
            s5[1] = mn;
            s5[2] = mx;
            s5[3] = c.cumsum[(size_t)iter][(size_t)q];
            s5[4] = c.cols;
        }
    });
}

SPS_API sps_status sps_fdmt_get_output_shape(const sps_fdmt* h, int64_t* rows, int64_t* cols) {
    return guarded([&] {
        SPS_REQUIRE(h && rows && cols, "null argument");
        *rows = h->eng.out_rows;
        *cols = h->eng.nsamps;
    });
}

SPS_API sps_status sps_fdmt_get_dt_grid_final(const sps_fdmt* h, int64_t* outv, int64_t cap, int64_t* n) {
    return guarded([&] {
        SPS_REQUIRE(h && n, "null argument");
        std::vector<int64_t> g;
        if (h->plan) g = h->plan->dt_grid_final();
        else
            for (int i = 0; i < h->cplan->imaxdt; ++i) g.push_back(i);
        *n = (int64_t)g.size();
        if (outv) std::copy(g.begin(), g.begin() + std::min<int64_t>(cap, (int64_t)g.size()), outv);
    });
}

SPS_API sps_status sps_fdmt_get_dm_grid_final(const sps_fdmt* h, float* outv, int64_t cap, int64_t* n) {
    return guarded([&] {
        SPS_REQUIRE(h && n, "null argument");
        SPS_REQUIRE(h->plan, "DM grid is defined for plan-based FDMT handles");
        auto g = h->plan->dm_grid_final();
        *n = (int64_t)g.size();
        if (outv) std::copy(g.begin(), g.begin() + std::min<int64_t>(cap, (int64_t)g.size()), outv);
    });
}

SPS_API sps_status sps_fdmt_get_df(const sps_fdmt* h, float* df, float* corr) {
    return guarded([&] {
        SPS_REQUIRE(h && df && corr, "null argument");
        SPS_REQUIRE(h->plan, "df is defined for plan-based FDMT handles");
        *df = h->plan->df;
        *corr = h->plan->correction;
    });
}

SPS_API sps_status sps_fdmt_get_plan_iter(const sps_fdmt* h, int64_t iter, int64_t* nsub, int64_t* grid_off,
                                          int64_t* grid, int64_t* nmap, int64_t* map7, int64_t* ncopy,
                                          int64_t* copy4, float* df_top, float* df_bot) {
    return guarded([&] {
        SPS_REQUIRE(h, "null handle");
        SPS_REQUIRE(h->plan, "plan tables are defined for plan-based FDMT handles");
        SPS_REQUIRE(iter >= 0 && iter <= h->plan->niters, "iteration out of range");
        const IterPlan& it = h->plan->iters[(size_t)iter];
        if (nsub) *nsub = it.nsub();
        if (grid_off) {
            grid_off[0] = 0;
            for (int64_t s = 0; s < it.nsub(); ++s) grid_off[s + 1] = grid_off[s] + (int64_t)it.dt_grid[(size_t)s].size();
        }
        if (grid) {
            int64_t k = 0;
            for (const auto& g : it.dt_grid)
                for (auto v : g) grid[k++] = v;
        }
        if (nmap) *nmap = (int64_t)it.maps.size();
        if (map7)
            for (size_t k = 0; k < it.maps.size(); ++k) {
                const Mapping& m = it.maps[k];
                int64_t* r = map7 + 7 * k;
                r[0] = m.out.sub; r[1] = m.out.dt; r[2] = m.head.sub; r[3] = m.head.dt;
                r[4] = m.tail.sub; r[5] = m.tail.dt; r[6] = m.offset;
            }
        if (ncopy) *ncopy = (int64_t)it.copies.size();
        if (copy4)
            for (size_t k = 0; k < it.copies.size(); ++k) {
                const Mapping& m = it.copies[k];
                int64_t* r = copy4 + 4 * k;
                r[0] = m.out.sub; r[1] = m.out.dt; r[2] = m.tail.sub; r[3] = m.tail.dt;
            }
        if (df_top) *df_top = it.df_top;
        if (df_bot) *df_bot = it.df_bot;
    });
}

SPS_API sps_status sps_fdmt_get_rows(const sps_fdmt* h, int64_t iter, int64_t* n, int64_t* rows4) {
    return guarded([&] {
        SPS_REQUIRE(h && n, "null argument");
        SPS_REQUIRE(iter >= 1 && iter <= h->eng.niters, "iteration out of range");
        const auto& rd = h->eng.iter[(size_t)iter];
        *n = (int64_t)rd.size();
        if (rows4)
            for (size_t k = 0; k < rd.size(); ++k) {
                rows4[4 * k + 0] = rd[k].out_row;
                rows4[4 * k + 1] = rd[k].tail_row;
                rows4[4 * k + 2] = rd[k].head_row;
                rows4[4 * k + 3] = rd[k].offset;
            }
    });
}

SPS_API sps_status sps_fdmt_execute(sps_fdmt* h, const void* d_wf, int dtype, size_t wf_size, float* d_dmt,
                                    size_t dmt_size, int ones, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(h, "null handle");
        const EnginePlan& e = h->eng;
        if (!ones) {
            SPS_REQUIRE(d_wf, "null waterfall");
            if ((int64_t)wf_size != e.nchans * e.nsamps) throw Error(SPS_ERR_INVALID_ARGUMENT, "Invalid size of waterfall");
        }
        SPS_REQUIRE(dtype == SPS_F32 || dtype == SPS_U8, "unknown dtype");
        SPS_REQUIRE(d_dmt, "null dmt");
        if ((int64_t)dmt_size != e.out_rows * e.nsamps) throw Error(SPS_ERR_INVALID_ARGUMENT, "Invalid size of dmt");
        if (e.niters > 0) h->check_channels(ones != 0);
        hipStream_t st = as_stream(stream);
        h->prepare(st);
        h->ensure_states(st);
        h->run(d_wf, dtype == SPS_U8, ones, e.nsamps, nullptr, e.nsamps, d_dmt, e.nsamps, h->state_a.as<float>(),
               h->state_b.as<float>(), h->pitch, st);
    });
}

SPS_API sps_status sps_fdmt_initialise(sps_fdmt* h, const void* d_wf, int dtype, float* d_state, size_t state_size,
                                       void* stream) {
    return guarded([&] {
        SPS_REQUIRE(h && d_wf && d_state, "null argument");
        const EnginePlan& e = h->eng;
        SPS_REQUIRE((int64_t)state_size == e.rows[0] * e.nsamps, "Invalid size of state");
        hipStream_t st = as_stream(stream);
        h->ensure_device(st);
        launch_fdmt_init(e.init_mode, d_wf, dtype == SPS_U8, 0, e.nsamps, nullptr, e.nchans, e.nsamps,
                         h->d_grid.as<int32_t>(), h->d_grid_off.as<int64_t>(), h->d_chan_row_off.as<int64_t>(), d_state,
                         e.nsamps, st, h->dmax, nullptr, h->grid_consec);
    });
}

SPS_API sps_status sps_fdmt_execute_host(sps_fdmt* h, const float* h_waterfall, size_t waterfall_size, float* h_dmt,
                                         size_t dmt_size, int ones) {
    return guarded([&] {
        SPS_REQUIRE(h && h_dmt, "null argument");
        const EnginePlan& e = h->eng;
        if (!ones) {
            SPS_REQUIRE(h_waterfall, "null waterfall");
            if ((int64_t)waterfall_size != e.nchans * e.nsamps)
                throw Error(SPS_ERR_INVALID_ARGUMENT, "Invalid size of waterfall");
        }
        if ((int64_t)dmt_size != e.out_rows * e.nsamps) throw Error(SPS_ERR_INVALID_ARGUMENT, "Invalid size of dmt");
        if (e.niters > 0) h->check_channels(ones != 0);
        hipStream_t st = nullptr;
        h->prepare(st);
        h->ensure_states(st);
        const void* d_in = nullptr;
        if (!ones) {
            h->host_in.ensure(sizeof(float) * waterfall_size);
            SPS_HIP(hipMemcpyAsync(h->host_in.p, h_waterfall, sizeof(float) * waterfall_size, hipMemcpyHostToDevice,
                                   st));
            d_in = h->host_in.p;
        }
        h->host_out.ensure(sizeof(float) * dmt_size);
        h->run(d_in, 0, ones, e.nsamps, nullptr, e.nsamps, h->host_out.as<float>(), e.nsamps, h->state_a.as<float>(),
               h->state_b.as<float>(), h->pitch, st);
        SPS_HIP(hipMemcpyAsync(h_dmt, h->host_out.p, sizeof(float) * dmt_size, hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
    });
}

SPS_API sps_status sps_fdmt_initialise_host(sps_fdmt* h, const float* h_waterfall, float* h_state, size_t state_size) {
    return guarded([&] {
        SPS_REQUIRE(h && h_waterfall && h_state, "null argument");
        const EnginePlan& e = h->eng;
        SPS_REQUIRE((int64_t)state_size == e.rows[0] * e.nsamps, "Invalid size of state");
        hipStream_t st = nullptr;
        h->ensure_device(st);
        const size_t nwf = (size_t)(e.nchans * e.nsamps);
        h->host_in.ensure(sizeof(float) * nwf);
        h->host_out.ensure(sizeof(float) * state_size);
        SPS_HIP(hipMemcpyAsync(h->host_in.p, h_waterfall, sizeof(float) * nwf, hipMemcpyHostToDevice, st));
        launch_fdmt_init(e.init_mode, h->host_in.p, 0, 0, e.nsamps, nullptr, e.nchans, e.nsamps,
                         h->d_grid.as<int32_t>(), h->d_grid_off.as<int64_t>(), h->d_chan_row_off.as<int64_t>(),
                         h->host_out.as<float>(), e.nsamps, st, h->dmax, nullptr, h->grid_consec);
        SPS_HIP(hipMemcpyAsync(h_state, h->host_out.p, sizeof(float) * state_size, hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
    });
}

SPS_API sps_status sps_cfdmt_get_config(const sps_fdmt* h, int64_t iter, int32_t* h_quant, int32_t* h_rows_cumsum,
                                        float* h_freq) {
    return guarded([&] {
        SPS_REQUIRE(h && h_quant, "null argument");
        SPS_REQUIRE(h->cplan, "not a legacy CFdmt handle");
        const CFdmtPlan& c = *h->cplan;
        SPS_REQUIRE(iter >= 0 && iter <= c.niter, "iteration out of range");
        const int q = c.quant[(size_t)iter];
        *h_quant = q;
        for (int k = 0; k <= q; ++k) {
            if (h_rows_cumsum) h_rows_cumsum[k] = c.cumsum[(size_t)iter][(size_t)k];
            if (h_freq) h_freq[k] = c.freq[(size_t)iter][(size_t)k];
        }
    });
}

SPS_API sps_status sps_fdmt_adjoint(sps_fdmt* h, const float* g_dmt, size_t dmt_size, float* g_wf, size_t wf_size,
                                    void* stream) {
    return guarded([&] {
        SPS_REQUIRE(h && g_dmt && g_wf, "null argument");
        const EnginePlan& e = h->eng;
        SPS_REQUIRE(e.init_mode != kInitRestrict, "the restrict init form is not linear; no adjoint");
        SPS_REQUIRE((int64_t)dmt_size == e.out_rows * e.nsamps, "Invalid size of dmt");
        SPS_REQUIRE((int64_t)wf_size == e.nchans * e.nsamps, "Invalid size of waterfall");
        SPS_REQUIRE(e.rows.back() == e.out_rows, "adjoint needs the full final state");
        hipStream_t st = as_stream(stream);
        h->ensure_device(st);
        h->build_adjoint(st);
        const int64_t N = e.nsamps, P = h->pitch;
        const float* cur = g_dmt;
        int64_t cur_pitch = N;
        for (size_t k = 0; k < h->adj.size(); ++k) {
            const auto& p = *h->adj[k];
            float* dst = (h->adj_shared ? (k % 2 ? h->state_b : h->state_a) : (k % 2 ? h->adj_b : h->adj_a)).as<float>();
            launch_fdmt_merge_adjoint(cur, cur_pitch, dst, P, p.depth, p.off.as<int64_t>(), p.users.as<AdjUser>(),
                                      p.prev_rows, N, st);
            cur = dst;
            cur_pitch = P;
        }
        launch_fdmt_init_adjoint(cur, cur_pitch, g_wf, N, e.nchans, N, h->d_grid.as<int32_t>(),
                                 h->d_grid_off.as<int64_t>(), h->d_chan_row_off.as<int64_t>(), h->dmax, st);
    });
}

// ---------------------------------------------------------------------------
// normalisation
// ---------------------------------------------------------------------------
SPS_API sps_status sps_calc_fdmt_inputs(float* d_in, int64_t nrows, int64_t ncols, float* d_buff, float* d_norm_input,
                                        int mode, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_in && nrows > 0 && ncols > 0, "invalid input");
        SPS_REQUIRE(mode == SPS_NORM_GLOBAL || mode == SPS_NORM_PER_CHANNEL, "mode must be global or per-channel");
        hipStream_t st = as_stream(stream);
        Arena m;
        const size_t rm = m.add<double>(nrows), rv = m.add<double>(nrows), stats = m.add<double>(8),
                     mu = m.add<float>(nrows), sg = m.add<float>(nrows), keep = m.add<uint8_t>(nrows);
        m.allocate();
        launch_row_stats(d_in, 0, nrows, ncols, m.at<double>(rm), m.at<double>(rv), st);
        launch_stats_finalize(m.at<double>(rm), m.at<double>(rv), nrows, mode, m.at<double>(stats), m.at<float>(mu),
                              m.at<float>(sg), m.at<uint8_t>(keep), d_buff, st);
        launch_apply_norm(d_in, d_norm_input, nrows, ncols, m.at<float>(mu), m.at<float>(sg), m.at<uint8_t>(keep), st);
        SPS_HIP(hipStreamSynchronize(st));
        m.idle();
    });
}

SPS_API sps_status sps_fdmt_normalization(const float* d_arr, const float* d_norm, int64_t len, float* d_out,
                                          void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_arr && d_norm && d_out && len >= 0, "invalid argument");
        launch_fdmt_normalization(d_arr, d_norm, len, d_out, as_stream(stream));
    });
}

SPS_API sps_status sps_fdmt_normalization_rows(const float* d_arr, int64_t rows, int64_t cols, const float* d_norm,
                                               int64_t norm_cols, float* d_out, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_arr && d_norm && d_out && rows >= 0 && cols >= 0, "invalid argument");
        SPS_REQUIRE(norm_cols >= 1 && norm_cols <= cols, "norm_cols must lie in 1..cols");
        launch_fdmt_normalization_rows(d_arr, rows, cols, d_norm, norm_cols, d_out, as_stream(stream));
    });
}

// ---------------------------------------------------------------------------
// candidates
// ---------------------------------------------------------------------------
}  // extern "C"

namespace {

template <typename K>
void sort_cands_k(CandD* c, int64_t n, int bt, int bw, int bits, hipStream_t st) {
    Arena m;
    const size_t k = m.add<K>(n), kt = m.add<K>(n), v = m.add<uint32_t>(n), vt = m.add<uint32_t>(n),
                 sc = m.add<uint8_t>((int64_t)sort_scratch_bytes(n));
    m.allocate();
    launch_cand_keys(c, n, bt, bw, m.at<K>(k), m.at<uint32_t>(v), m.at<void>(sc), st);
    const bool sw = radix_sort_pairs(m.at<K>(k), m.at<uint32_t>(v), m.at<K>(kt), m.at<uint32_t>(vt), n, bits,
                                     m.at<void>(sc), st);
    launch_cand_from_keys(m.at<K>(sw ? kt : k), m.at<uint32_t>(sw ? vt : v), n, bt, bw, c, st);
    SPS_HIP(hipStreamSynchronize(st));
    m.idle();
}

// Sorts n candidates in place by (mdt, mt, mwidth).
void sort_cands(CandD* c, int64_t n, int64_t rows, int64_t cols, int64_t wmax, hipStream_t st) {
    if (n <= 1) return;
    const int bt = std::max(1, bitlen((uint64_t)cols)), bw = std::max(1, bitlen((uint64_t)wmax)),
              br = std::max(1, bitlen((uint64_t)rows));
    SPS_REQUIRE(bt + bw + br <= 64, "candidate key does not fit 64 bits");
    // mt < cols, mdt < rows: one bit less each where those are powers of two
    const int t = std::max(1, bitlen((uint64_t)cols - 1)), r = std::max(1, bitlen((uint64_t)rows - 1));
    if (t + bw + r <= 32) sort_cands_k<uint32_t>(c, n, t, bw, t + bw + r, st);
    else sort_cands_k<uint64_t>(c, n, t, bw, t + bw + r, st);
}

// Every candidate of the image, sorted by (mdt, mt, mwidth), into `out`
// (a DevBuf or ScratchBuf, grown to the count); returns the count.  The first
// pass finds room for a megabyte's worth, so that only larger counts gather
// twice.  Synchronises st.
template <class Buf>
int64_t gather_sorted(const float* img, int64_t rows, int64_t cols, int64_t pitch, const float* d_thr, float h_thr,
                      int wnd, bool pow2, Buf& out, Buf& cnt, hipStream_t st) {
    const int64_t wmax = pow2 ? (int64_t)1 << wnd : wnd;
    cnt.ensure(sizeof(unsigned long long));
    out.ensure((size_t)1 << 20);
    int64_t tcap = (int64_t)(out.bytes / sizeof(CandD));
    unsigned long long n = 0;
    for (int pass = 0; pass < 2; ++pass) {
        launch_fill_u64(cnt.template as<unsigned long long>(), 1, 0ull, st);
        launch_boxcar(img, rows, cols, pitch, d_thr, h_thr, (int)wmax, pow2, out.template as<CandD>(), tcap,
                      cnt.template as<unsigned long long>(), st);
        SPS_HIP(hipMemcpyAsync(&n, cnt.p, sizeof(n), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        if ((int64_t)n <= tcap) break;
        tcap = (int64_t)n;
        out.ensure(sizeof(CandD) * (size_t)tcap);
    }
    sort_cands(out.template as<CandD>(), (int64_t)n, rows, cols, pow2 ? wnd : wmax, st);
    return (int64_t)n;
}

// Below this many candidates a level's keys take the width that any number of
// groups fits: reading the count back costs about two passes of the sort.
constexpr int64_t kClusterReadback = 1 << 16;

// Three-key gap clustering (Clusterization.cu:92-166) of n candidates with the
// device bins, delegates sorted by mt into d_delegates / d_group_size;
// returns the group count.  Synchronises st.
int64_t cluster_candidates(const CandD* c, int64_t n, const int32_t* d_bins, int32_t* d_delegates,
                           int64_t* d_group_size, hipStream_t st) {
    if (n == 0) return 0;
    SPS_REQUIRE(n < 0xffffffffLL, "invalid candidate count");
    Arena m;
    const size_t k = m.add<uint64_t>(n), kt = m.add<uint64_t>(n), v = m.add<uint32_t>(n), vt = m.add<uint32_t>(n),
                 grp = m.add<uint32_t>(n), flags = m.add<uint32_t>(n), sc = m.add<uint8_t>((int64_t)sort_scratch_bytes(n)),
                 rg = m.add<uint32_t>(6), best = m.add<unsigned long long>(n), start = m.add<uint32_t>(n);
    m.allocate();
    uint32_t ranges[6];
    size_t perm = v;
    uint32_t ng = 1;  // groups of the level before, at most
    if (launch_cluster_small(c, n, d_bins, m.at<uint32_t>(v), m.at<uint32_t>(flags), m.at<uint32_t>(grp),
                             m.at<uint32_t>(rg), st)) {
        SPS_HIP(hipMemcpyAsync(ranges, m.at<void>(rg), 3 * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        ng = ranges[2];
    } else {
        launch_fill_u64(m.at<unsigned long long>(rg), 3, 0xffffffffull, st);  // {0xffffffff, 0} three times
        launch_cand_ranges(c, n, m.at<uint32_t>(rg), st);
        SPS_HIP(hipMemcpyAsync(ranges, m.at<void>(rg), sizeof(ranges), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        for (int level = 0; level < 3; ++level) {
            const uint32_t base = ranges[2 * level];
            const int bm = bitlen(ranges[2 * level + 1] - base), bits = bm + (level ? bitlen(ng) : 0);
            const uint32_t* p = level ? m.at<uint32_t>(perm) : nullptr;
            const uint32_t* g = level ? m.at<uint32_t>(grp) : nullptr;
            const size_t vin = level && perm == v ? vt : v, vtmp = vin == v ? vt : v;
            auto run = [&](auto key) {
                using K = decltype(key);
                launch_cluster_keys(c, p, g, n, level, base, bm, m.at<K>(k), m.at<uint32_t>(vin), m.at<void>(sc), st);
                const bool sw = radix_sort_pairs(m.at<K>(k), m.at<uint32_t>(vin), m.at<K>(kt), m.at<uint32_t>(vtmp), n,
                                                 bits, m.at<void>(sc), st);
                perm = sw ? vtmp : vin;
                launch_cluster_groups(m.at<K>(sw ? kt : k), n, bm, d_bins, level, m.at<void>(sc),
                                      m.at<uint32_t>(flags), m.at<uint32_t>(grp), st);
            };
            if (bits <= 32) run(uint32_t{});
            else run(uint64_t{});
            ng = (uint32_t)n;
            if (level == 2 || n >= kClusterReadback) {
                SPS_HIP(hipMemcpyAsync(&ng, m.at<uint32_t>(grp) + (n - 1), sizeof(uint32_t), hipMemcpyDeviceToHost,
                                       st));
                SPS_HIP(hipStreamSynchronize(st));
            }
        }
    }
    launch_fill_u64(m.at<unsigned long long>(best), ng, 0ull, st);
    launch_cluster_delegates(c, m.at<uint32_t>(perm), m.at<uint32_t>(grp), m.at<uint32_t>(flags), n,
                             m.at<unsigned long long>(best), m.at<uint32_t>(start), st);
    // (the permutation is no longer needed)
    launch_delegate_keys(c, m.at<unsigned long long>(best), ng, ranges[0], m.at<uint32_t>(k), m.at<uint32_t>(v),
                         m.at<void>(sc), st);
    const bool sw = radix_sort_pairs(m.at<uint32_t>(k), m.at<uint32_t>(v), m.at<uint32_t>(kt), m.at<uint32_t>(vt), ng,
                                     bitlen(ranges[1] - ranges[0]), m.at<void>(sc), st);
    launch_delegate_out(m.at<unsigned long long>(best), m.at<uint32_t>(start), m.at<uint32_t>(sw ? vt : v), ng, n,
                        d_delegates, d_group_size, st);
    SPS_HIP(hipStreamSynchronize(st));
    m.idle();
    return (int64_t)ng;
}

}  // namespace

extern "C" {

SPS_API sps_status sps_boxcar_candidates(const float* d_img, int64_t rows, int64_t cols, const float* d_thr, int wnd,
                                         int all_widths, sps_cand* d_out, int64_t cap, int64_t* h_count,
                                         void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_img && d_thr && h_count, "null argument");
        SPS_REQUIRE(rows > 0 && cols > 0 && cap >= 0, "invalid sizes");
        SPS_REQUIRE(cap == 0 || d_out, "null output");
        const bool pow2 = !all_widths;
        SPS_REQUIRE(wnd >= (pow2 ? 0 : 1) && wnd <= (pow2 ? 13 : 8192), "window parameter out of range");
        hipStream_t st = as_stream(stream);
        ScratchBuf cnt, tmp;
        const int64_t n = gather_sorted(d_img, rows, cols, cols, d_thr, 0.f, wnd, pow2, tmp, cnt, st);
        const int64_t ncopy = std::min<int64_t>(n, cap);
        if (ncopy > 0)
            SPS_HIP(hipMemcpyAsync(d_out, tmp.p, sizeof(CandD) * (size_t)ncopy, hipMemcpyDeviceToDevice, st));
        SPS_HIP(hipStreamSynchronize(st));
        cnt.idle();
        tmp.idle();
        *h_count = n;
        if (n > cap) throw Error(SPS_ERR_CAPACITY, "more candidates than the output capacity");
    });
}

SPS_API sps_status sps_cluster(const sps_cand* d_cands, int64_t n, const int32_t* d_bins, int32_t* d_delegates,
                               int64_t* d_group_size, int64_t* h_ngroups, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(h_ngroups && d_bins, "null argument");
        SPS_REQUIRE(n >= 0 && n < 0xffffffffLL, "invalid candidate count");
        *h_ngroups = 0;
        if (n == 0) return;
        SPS_REQUIRE(d_cands && d_delegates && d_group_size, "null argument");
        *h_ngroups = cluster_candidates(reinterpret_cast<const CandD*>(d_cands), n, d_bins, d_delegates, d_group_size,
                                        as_stream(stream));
    });
}

SPS_API sps_status sps_detect_max(const float* d_arr, const float* d_norm, int64_t rows, int64_t cols, int wnd,
                                  sps_detection* d_out, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_arr && d_out && rows > 0 && cols > 0 && wnd >= 1, "invalid argument");
        hipStream_t st = as_stream(stream);
        ScratchBuf blocks;
        const int64_t nb = detect_max_blocks(rows, cols);
        blocks.ensure(16 * (size_t)nb);
        launch_detect_max(d_arr, d_norm, rows, cols, wnd, blocks.p, nb, d_out, st);
        SPS_HIP(hipStreamSynchronize(st));
        blocks.idle();
    });
}

SPS_API sps_status sps_boxcar_snr(const float* d_img, int64_t rows, int64_t cols, int w, float* d_snr, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_img && d_snr && rows > 0 && cols > 0 && w >= 1, "invalid argument");
        launch_boxcar_snr(d_img, rows, cols, w, d_snr, as_stream(stream));
    });
}

SPS_API sps_status sps_digitize(float* d_x, int64_t n, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(n >= 0 && (d_x || n == 0), "invalid argument");
        launch_digitize(d_x, n, as_stream(stream));
    });
}

SPS_API sps_status sps_boxcar_snr_adjoint(const float* d_g, int64_t rows, int64_t cols, int w, float* d_gi,
                                          void* stream) {
    return guarded([&] {
        SPS_REQUIRE(d_g && d_gi && rows > 0 && cols > 0 && w >= 1, "invalid argument");
        launch_boxcar_snr_adjoint(d_g, rows, cols, w, d_gi, as_stream(stream));
    });
}

}  // extern "C"

// ---------------------------------------------------------------------------
// fused single-beam search
// ---------------------------------------------------------------------------
struct sps_search {
    sps_search_params p{};
    std::unique_ptr<sps_fdmt> f;     // data transform (nsamps)
    int64_t ndt = 0;
    int64_t norm_len = 0;            // samples of the mask transform
    DevBuf rm, rv, stats, mu, sg, keep, zeros, ones_f;
    DevBuf norm_img, norm_a, norm_b; // mask transform output and its states
    DevBuf mask_shift;               // [ndt][nchans] int16 channel shifts (empty: run the transform)
    DevBuf dmt;                      // internal DM-time image when the caller passes none
    bool ready = false;
    // clustering leg (sps_search_cluster): all-widths candidates, delegates
    DevBuf heap, heap_cnt, d_del, d_gsz;
    int64_t heap_n = 0;
    std::vector<int32_t> h_del;
    std::vector<int64_t> h_gsz;
    std::vector<sps_cand> h_del_cand;  // the delegates' candidates
    // stage timing: ev[0] start, ev[1] stats, ev[2..] init + merges, then
    // mask transform, S/N normalisation, boxcar
    bool timing = false;
    std::vector<hipEvent_t> ev;

    ~sps_search() {
        for (auto e : ev) (void)hipEventDestroy(e);
    }
    // stats, mask transform, init, one per pass, separate S/N, boxcar
    int64_t nstages() const { return (int64_t)f->schedule.size() + 5; }
    void ensure_events() {
        const size_t need = (size_t)nstages() + 1;
        while (ev.size() < need) {
            hipEvent_t e;
            SPS_HIP(hipEventCreate(&e));
            ev.push_back(e);
        }
    }

    // device scratch of one search (floats): ping-pong states, mask transform
    // states and image, and the DM-time image when the caller passes none.
    // A batch hands one set, sized for the largest of its beams, to every
    // beam that runs on the same stream.
    struct Scratch {
        float *sa = nullptr, *sb = nullptr, *na = nullptr, *nb = nullptr, *nimg = nullptr, *dmt = nullptr;
    };
    struct ScratchSize {
        int64_t sa = 0, sb = 0, na = 0, nb = 0, nimg = 0, dmt = 0;
    };
    ScratchSize scratch_size() const {
        ScratchSize z;
        int64_t ra, rb;
        f->state_rows(ra, rb);
        z.sa = checked_mul(ra, f->pitch, "state");
        z.sb = checked_mul(rb, f->pitch, "state");
        if (p.snr_norm) {
            const int64_t Pn = round_up(norm_len, 4);
            if (!mask_shift.p) {
                z.na = checked_mul(ra, Pn, "norm");
                z.nb = checked_mul(rb, Pn, "norm");
            }
            z.nimg = checked_mul(ndt, norm_len, "norm");
        }
        z.dmt = checked_mul(ndt, p.nsamps, "dmt");
        return z;
    }

    void setup(hipStream_t st, bool own_scratch = true) {
        if (!ready) setup_small(st);
        f->prepare(st);
        if (own_scratch) {
            f->ensure_states(st);
            if (p.snr_norm) {
                const ScratchSize z = scratch_size();
                norm_img.ensure(sizeof(float) * (size_t)z.nimg);
                norm_a.ensure(sizeof(float) * (size_t)z.na);
                norm_b.ensure(sizeof(float) * (size_t)z.nb);
            }
        }
    }

    Scratch own_scratch() {
        Scratch s;
        s.sa = f->state_a.as<float>();
        s.sb = f->state_b.as<float>();
        s.na = norm_a.as<float>();
        s.nb = norm_b.as<float>();
        s.nimg = norm_img.as<float>();
        return s;
    }

    // per-search tables and statistics buffers (small)
    void setup_small(hipStream_t st) {
        const int64_t R = p.nchans;
        rm.ensure(sizeof(double) * (size_t)R);
        rv.ensure(sizeof(double) * (size_t)R);
        stats.ensure(sizeof(double) * 8);
        mu.ensure(sizeof(float) * (size_t)R);
        sg.ensure(sizeof(float) * (size_t)R);
        keep.ensure((size_t)R);
        std::vector<float> z((size_t)R, 0.f), o((size_t)R, 1.f);
        upload(zeros, z, st);
        upload(ones_f, o, st);
        if (p.norm_mode == SPS_NORM_NONE) {
            // no cleaning: every channel kept, unit scale, mask of ones
            std::vector<uint8_t> k((size_t)R, 1);
            upload(keep, k, st);
            upload(mu, z, st);
            upload(sg, o, st);
            std::vector<double> s = {0.0, 1.0, 0.0, 0.0, (double)R, 0.0, 0.0, 0.0};
            upload(stats, s, st);
        }
        SPS_HIP(hipStreamSynchronize(st));
        ready = true;
    }

    // Enqueues one beam on st (no host synchronisation, no allocation, no
    // memset: safe under stream capture once setup() has run).
    void enqueue(const void* d_in, float* d_dmt, sps_cand* d_cands, uint64_t* d_count, hipStream_t st,
                 const Scratch& sc, hipEvent_t* ev) {
        const int64_t N = p.nsamps;
        const int it = (int)f->schedule.size();  // passes
        if (ev) SPS_HIP(hipEventRecord(ev[0], st));
        if (p.norm_mode != SPS_NORM_NONE) {
            launch_row_stats(d_in, p.in_dtype == SPS_U8, p.nchans, N, rm.as<double>(), rv.as<double>(), st);
            launch_stats_finalize(rm.as<double>(), rv.as<double>(), p.nchans, p.norm_mode, stats.as<double>(),
                                  mu.as<float>(), sg.as<float>(), keep.as<uint8_t>(), nullptr, st,
                                  reinterpret_cast<unsigned long long*>(d_count));
        }
        if (ev) SPS_HIP(hipEventRecord(ev[1], st));
        float* out = d_dmt ? d_dmt : sc.dmt;
        SPS_REQUIRE(out, "no DM-time image buffer");
        // mask transform first: its output feeds the S/N epilogue of the last merge
        MergeEpilogue epi{nullptr, 0, nullptr};
        const bool fuse = p.snr_norm && f->eng.niters > 0;
        if (p.snr_norm) {
            const int64_t L = norm_len;
            if (mask_shift.p) {
                launch_mask_counts(mask_shift.as<int16_t>(), keep.as<uint8_t>(), ndt, p.nchans, (int)L, sc.nimg, L,
                                   st);
            } else {
                ChanNorm mask{zeros.as<float>(), ones_f.as<float>(), keep.as<uint8_t>()};
                f->run(nullptr, 0, 1, N, &mask, L, sc.nimg, L, sc.na, sc.nb, round_up(L, 4), st, nullptr, nullptr,
                       true);
            }
            epi = MergeEpilogue{sc.nimg, L, stats.as<double>()};
        }
        if (ev) SPS_HIP(hipEventRecord(ev[2], st));
        ChanNorm cn{mu.as<float>(), sg.as<float>(), keep.as<uint8_t>()};
        const ChanNorm* np = (p.norm_mode != SPS_NORM_NONE) ? &cn : nullptr;
        f->run(d_in, p.in_dtype == SPS_U8, 0, N, np, N, out, N, sc.sa, sc.sb, f->pitch, st, ev ? ev + 3 : nullptr,
               fuse ? &epi : nullptr);
        if (p.snr_norm && !fuse)
            launch_snr_normalise(out, ndt, N, N, sc.nimg, norm_len, stats.as<double>(), st);
        if (ev) SPS_HIP(hipEventRecord(ev[it + 4], st));
        if (p.norm_mode == SPS_NORM_NONE) launch_fill_u64(reinterpret_cast<unsigned long long*>(d_count), 1, 0ull, st);
        launch_boxcar(out, ndt, N, N, nullptr, p.threshold, 1 << p.box_q, 1, reinterpret_cast<CandD*>(d_cands),
                      p.cand_capacity, reinterpret_cast<unsigned long long*>(d_count), st);
        if (ev) SPS_HIP(hipEventRecord(ev[it + 5], st));
    }
};

// The mask transform's input is 1 on every sample of a kept channel and 0
// elsewhere.  With the running-mean init its cells are exactly 1 from t = the
// cell's dt on and 0 before (a mean of ones; cells t < dt are zero), and each
// merge adds exact small integers, a head counted from t = offset on.  So
// output row r at t counts
// the kept channels whose accumulated shift along r's tree (init dt plus the
// head offsets on the path) is <= t.  The shifts are tabulated here per
// (output row, channel); a row that would hold a channel twice, or shifts
// beyond int16, leave the table empty and the transform runs instead, as it
// does for the legacy plans.
static void build_mask_shifts(sps_search& s) {
    const EnginePlan& e = s.f->eng;
    const int64_t L = s.norm_len;
    const int64_t R = e.out_rows, C = e.nchans;
    // (L, rounded up to 4) LDS counters within 64 KiB
    if (e.init_mode != kInitMean || L <= 0 || L > 16000 || R <= 0 || C <= 0 || R * C > ((int64_t)1 << 31)) return;
    // state-0 row -> channel and init dt
    std::vector<int32_t> chan0((size_t)e.rows[0], -1), dt0((size_t)e.rows[0], 0);
    for (int64_t c = 0; c < C; ++c)
        for (int64_t k = e.grid_off[(size_t)c]; k < e.grid_off[(size_t)c + 1]; ++k) {
            const int64_t r0 = e.chan_row_off[(size_t)c] + (k - e.grid_off[(size_t)c]);
            chan0[(size_t)r0] = (int32_t)c;
            dt0[(size_t)r0] = e.grid[(size_t)k];
        }
    // per iteration: output row -> its record
    std::vector<std::vector<int64_t>> rec((size_t)e.niters + 1);
    for (int i = 1; i <= e.niters; ++i) {
        rec[(size_t)i].assign((size_t)e.rows[(size_t)i], -1);
        const auto& it = e.iter[(size_t)i];
        for (size_t j = 0; j < it.size(); ++j) rec[(size_t)i][(size_t)it[j].out_row] = (int64_t)j;
    }
    std::vector<int16_t> tab((size_t)(R * C), (int16_t)32767);
    struct Node {
        int i;
        int64_t row, base;
    };
    std::vector<Node> stack;
    for (int64_t r = 0; r < R; ++r) {
        int16_t* trow = tab.data() + (size_t)(r * C);
        stack.assign(1, Node{e.niters, r, 0});
        while (!stack.empty()) {
            const Node n = stack.back();
            stack.pop_back();
            if (n.i == 0) {
                const int32_t c = chan0[(size_t)n.row];
                const int64_t sh = n.base + dt0[(size_t)n.row];
                if (c < 0 || trow[c] != 32767 || sh < 0 || sh >= 32767) return;  // unexpected: keep the transform
                trow[c] = (int16_t)sh;
                continue;
            }
            const int64_t j = rec[(size_t)n.i][(size_t)n.row];
            if (j < 0) return;
            const RowDesc& d = e.iter[(size_t)n.i][(size_t)j];
            stack.push_back(Node{n.i - 1, d.tail_row, n.base});
            if (d.head_row >= 0) stack.push_back(Node{n.i - 1, d.head_row, n.base + d.offset});
        }
    }
    s.mask_shift.ensure(sizeof(int16_t) * tab.size());
    SPS_HIP(hipMemcpy(s.mask_shift.p, tab.data(), sizeof(int16_t) * tab.size(), hipMemcpyHostToDevice));
}

// cfdmt_imaxdt > 0: the data transform is the legacy CFdmt plan
// (CFdmtGpu(f_min, f_max, nchans, nsamps, imaxDt)) instead of the FDMT plan;
// dt_max and tsamp are then unused
static std::unique_ptr<sps_search> make_search(const sps_search_params* p, int cfdmt_imaxdt = 0) {
    SPS_REQUIRE(p->in_dtype == SPS_F32 || p->in_dtype == SPS_U8, "unknown dtype");
    SPS_REQUIRE(p->norm_mode >= SPS_NORM_NONE && p->norm_mode <= SPS_NORM_PER_CHANNEL, "unknown norm mode");
    SPS_REQUIRE(p->box_q >= 0 && p->box_q <= 13, "box_q out of range");
    SPS_REQUIRE(p->cand_capacity >= 0, "negative capacity");
    std::unique_ptr<sps_search> s(new sps_search());
    s->p = *p;
    s->f.reset(new sps_fdmt());
    if (cfdmt_imaxdt > 0) {
        SPS_REQUIRE(p->nchans <= INT32_MAX && p->nsamps <= INT32_MAX, "CFdmt sizes must fit in int");
        s->f->cplan.reset(new CFdmtPlan(p->f_min, p->f_max, (int)p->nchans, (int)p->nsamps, cfdmt_imaxdt));
        s->f->eng = s->f->cplan->lower();
    } else {
        s->f->plan.reset(new FdmtPlan(p->f_min, p->f_max, p->nchans, p->nsamps, p->tsamp, p->dt_max, 1, 0));
        s->f->eng = s->f->plan->lower(kInitMean);
    }
    s->f->init_layout();
    s->ndt = s->f->eng.out_rows;
    // the mask transform is causal: samples t < L depend on inputs before
    // L only, and beyond the longest channel track every kept channel
    // contributes exactly 1, so the divisor there is the kept count
    const EnginePlan& e = s->f->eng;
    std::vector<int64_t> ext((size_t)e.rows[0]);
    for (int64_t c = 0; c < e.nchans; ++c)
        for (int64_t k = e.grid_off[(size_t)c]; k < e.grid_off[(size_t)c + 1]; ++k)
            ext[(size_t)(e.chan_row_off[(size_t)c] + (k - e.grid_off[(size_t)c]))] = e.grid[(size_t)k];
    for (int i = 1; i <= e.niters; ++i) {
        std::vector<int64_t> nx((size_t)e.rows[(size_t)i], 0);
        for (const auto& r : e.iter[(size_t)i]) {
            int64_t v = ext[(size_t)r.tail_row];
            if (r.head_row >= 0) v = std::max(v, ext[(size_t)r.head_row] + r.offset);
            nx[(size_t)r.out_row] = v;
        }
        ext.swap(nx);
    }
    int64_t mx = 0;
    for (auto v : ext) mx = std::max(mx, v);
    s->norm_len = std::min<int64_t>(p->nsamps, mx + 1);
    build_mask_shifts(*s);
    return s;
}

extern "C" {

SPS_API sps_status sps_search_create(const sps_search_params* p, sps_search** out) {
    return guarded([&] {
        SPS_REQUIRE(p && out, "null argument");
        *out = nullptr;
        *out = make_search(p).release();
    });
}

SPS_API sps_status sps_search_create_cfdmt(const sps_search_params* p, int imaxdt, sps_search** out) {
    return guarded([&] {
        SPS_REQUIRE(p && out, "null argument");
        SPS_REQUIRE(imaxdt >= 1, "imaxdt must be positive");
        *out = nullptr;
        *out = make_search(p, imaxdt).release();
    });
}

SPS_API sps_status sps_search_destroy(sps_search* s) {
    return guarded([&] {
        delete s;
        scratch_trim();
    });
}

SPS_API sps_status sps_search_get_ndt(const sps_search* s, int64_t* n) {
    return guarded([&] {
        SPS_REQUIRE(s && n, "null argument");
        *n = s->ndt;
    });
}

SPS_API sps_status sps_search_run(sps_search* s, const void* d_in, float* d_dmt, sps_cand* d_cands,
                                  uint64_t* d_count, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(s && d_in && d_count, "null argument");
        SPS_REQUIRE(s->p.cand_capacity == 0 || d_cands, "null candidate buffer");
        hipStream_t st = as_stream(stream);
        s->setup(st);
        sps_search::Scratch sc = s->own_scratch();
        if (!d_dmt) {
            s->dmt.ensure(sizeof(float) * (size_t)s->scratch_size().dmt);
            sc.dmt = s->dmt.as<float>();
        }
        hipEvent_t* ev = nullptr;
        if (s->timing) {
            s->ensure_events();
            ev = s->ev.data();
        }
        s->enqueue(d_in, d_dmt, d_cands, d_count, st, sc, ev);
    });
}

SPS_API sps_status sps_fdmt_set_schedule(sps_fdmt* h, const int32_t* h_depths, int64_t n) {
    return guarded([&] {
        SPS_REQUIRE(h && (n == 0 || h_depths), "null argument");
        h->set_schedule(std::vector<int>(h_depths, h_depths + n));
    });
}

SPS_API sps_status sps_fdmt_get_schedule(const sps_fdmt* h, int32_t* h_depths, int64_t cap, int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(h && h_n, "null argument");
        *h_n = (int64_t)h->schedule.size();
        for (int64_t i = 0; i < *h_n && i < cap && h_depths; ++i) h_depths[i] = h->schedule[(size_t)i];
    });
}

SPS_API sps_status sps_fdmt_set_staged(sps_fdmt* h, int staged) {
    return guarded([&] {
        SPS_REQUIRE(h, "null handle");
        h->set_staged(staged);
    });
}

SPS_API sps_status sps_search_set_staged(sps_search* s, int staged) {
    return guarded([&] {
        SPS_REQUIRE(s, "null handle");
        s->f->set_staged(staged);
    });
}

SPS_API sps_status sps_fdmt_set_group_shape(sps_fdmt* h, int lds_floats, int max_rows, int tiles_per_block) {
    return guarded([&] {
        SPS_REQUIRE(h, "null handle");
        h->set_group_shape(lds_floats, max_rows, tiles_per_block);
    });
}

SPS_API sps_status sps_search_set_group_shape(sps_search* s, int lds_floats, int max_rows, int tiles_per_block) {
    return guarded([&] {
        SPS_REQUIRE(s, "null handle");
        s->f->set_group_shape(lds_floats, max_rows, tiles_per_block);
    });
}

SPS_API sps_status sps_search_set_schedule(sps_search* s, const int32_t* h_depths, int64_t n) {
    return guarded([&] {
        SPS_REQUIRE(s && (n == 0 || h_depths), "null argument");
        s->f->set_schedule(std::vector<int>(h_depths, h_depths + n));
    });
}

SPS_API sps_status sps_search_get_schedule(const sps_search* s, int32_t* h_depths, int64_t cap, int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(s && h_n, "null argument");
        *h_n = (int64_t)s->f->schedule.size();
        for (int64_t i = 0; i < *h_n && i < cap && h_depths; ++i) h_depths[i] = s->f->schedule[(size_t)i];
    });
}

SPS_API sps_status sps_search_enable_timing(sps_search* s, int enable) {
    return guarded([&] {
        SPS_REQUIRE(s, "null handle");
        s->timing = enable != 0;
        if (s->timing) s->ensure_events();
    });
}

SPS_API sps_status sps_search_get_timing(sps_search* s, double* h_ms, int64_t cap, int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(s && h_n, "null argument");
        SPS_REQUIRE(s->timing, "timing is not enabled");
        const int64_t n = s->nstages();
        *h_n = n;
        SPS_HIP(hipEventSynchronize(s->ev[(size_t)n]));
        for (int64_t i = 0; i < n && i < cap; ++i) {
            float ms = 0.f;
            SPS_HIP(hipEventElapsedTime(&ms, s->ev[(size_t)i], s->ev[(size_t)i + 1]));
            h_ms[i] = ms;
        }
    });
}

SPS_API sps_status sps_search_get_stage_bytes(const sps_search* s, double* h_b, int64_t cap, int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(s && h_n, "null argument");
        const sps_fdmt& f = *s->f;
        const EnginePlan& e = f.eng;
        const double N = (double)s->p.nsamps, N4 = 4.0 * N;
        const double in_elem = s->p.in_dtype == SPS_U8 ? 1.0 : 4.0;
        const double in_bytes = in_elem * N * (double)e.nchans;
        std::vector<double> b;
        b.push_back(s->p.norm_mode != SPS_NORM_NONE ? in_bytes : 0.0);  // statistics: one input read
        // mask transform: its output image (ndt rows over its extent), written
        // once and read once by the final pass; its states stay in the caches
        b.push_back(s->p.snr_norm ? 2.0 * 4.0 * (double)s->norm_len * (double)s->ndt : 0.0);
        // init: input read + live state-0 rows; with the init fused into the
        // first pass, state 0 never reaches HBM and that pass reads the input
        b.push_back(f.ran_fused0 ? 0.0 : in_bytes + N4 * (double)f.live_rows(0));
        // a launch reads the live rows of the state before it and writes those
        // of its last; like its time, that counts for the first schedule
        // entry that ends with it
        const size_t entry0 = b.size();
        b.resize(entry0 + f.schedule.size(), 0.0);
        int i0 = 1, entry_end = 0;
        size_t done = 0;
        double bytes = 0.0;
        for (int L : f.pass_depths()) {
            const int top = i0 + L - 1;
            bytes += ((i0 == 1 && f.ran_fused0) ? in_bytes : N4 * (double)f.live_rows(i0 - 1)) + N4 * (double)f.live_rows(top);
            while (done < f.schedule.size() && entry_end + f.schedule[done] <= top) {
                entry_end += f.schedule[done];
                b[entry0 + done++] = bytes;
                bytes = 0.0;
            }
            i0 += L;
        }
        b.push_back(0.0);                                                // S/N normalisation (fused into the last pass)
        b.push_back(N4 * (double)s->ndt);                                // boxcar: one read of the image
        *h_n = (int64_t)b.size();
        for (int64_t i = 0; i < (int64_t)b.size() && i < cap; ++i) h_b[i] = b[(size_t)i];
    });
}

SPS_API sps_status sps_search_sort_candidates(sps_search* s, sps_cand* d_cands, const uint64_t* d_count,
                                              int64_t* h_count, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(s && d_count && h_count, "null argument");
        hipStream_t st = as_stream(stream);
        unsigned long long n = 0;
        SPS_HIP(hipMemcpyAsync(&n, d_count, sizeof(n), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        const int64_t m = std::min<int64_t>((int64_t)n, s->p.cand_capacity);
        sort_cands(reinterpret_cast<CandD*>(d_cands), m, s->ndt, s->p.nsamps, s->p.box_q, st);
        *h_count = (int64_t)n;
        // the kept prefix is whichever candidates won the counter first: the
        // caller must re-gather into a buffer of h_count entries
        if ((int64_t)n > s->p.cand_capacity)
            throw Error(SPS_ERR_CAPACITY, "more candidates than cand_capacity: re-gather with sps_search_gather");
    });
}

SPS_API sps_status sps_search_gather(sps_search* s, const float* d_dmt, sps_cand* d_cands, int64_t cap,
                                     uint64_t* d_count, int64_t* h_count, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(s && d_count && h_count && cap >= 0 && (cap == 0 || d_cands), "null argument");
        const float* img = d_dmt ? d_dmt : s->dmt.as<float>();
        SPS_REQUIRE(img, "no DM-time image: run the search first (or pass the image it wrote)");
        hipStream_t st = as_stream(stream);
        const int64_t N = s->p.nsamps;
        launch_fill_u64(reinterpret_cast<unsigned long long*>(d_count), 1, 0ull, st);
        launch_boxcar(img, s->ndt, N, N, nullptr, s->p.threshold, 1 << s->p.box_q, 1,
                      reinterpret_cast<CandD*>(d_cands), cap, reinterpret_cast<unsigned long long*>(d_count), st);
        unsigned long long n = 0;
        SPS_HIP(hipMemcpyAsync(&n, d_count, sizeof(n), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        sort_cands(reinterpret_cast<CandD*>(d_cands), std::min<int64_t>((int64_t)n, cap), s->ndt, N, s->p.box_q, st);
        *h_count = (int64_t)n;
        if ((int64_t)n > cap) throw Error(SPS_ERR_CAPACITY, "more candidates than the gather's capacity");
    });
}

SPS_API sps_status sps_search_cluster(sps_search* s, const float* d_dmt, int wnd, const int32_t* d_bins,
                                      int64_t* h_ncand, int64_t* h_ngroups, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(s && d_bins && h_ncand && h_ngroups, "null argument");
        SPS_REQUIRE(wnd >= 1 && wnd <= 8192, "window must be 1..8192");
        const float* img = d_dmt ? d_dmt : s->dmt.as<float>();
        SPS_REQUIRE(img, "no DM-time image: run the search first (or pass the image it wrote)");
        hipStream_t st = as_stream(stream);
        s->heap_n = 0;
        s->h_del.clear();
        s->h_gsz.clear();
        s->h_del_cand.clear();
        *h_ncand = 0;
        *h_ngroups = 0;
        const int64_t N = s->p.nsamps;
        const int64_t n = gather_sorted(img, s->ndt, N, N, nullptr, s->p.threshold, wnd, false, s->heap, s->heap_cnt, st);
        s->heap_n = n;
        *h_ncand = n;
        if (n == 0) return;
        s->d_del.ensure(sizeof(int32_t) * (size_t)n);
        s->d_gsz.ensure(sizeof(int64_t) * (size_t)n);
        const int64_t ng = cluster_candidates(s->heap.as<CandD>(), n, d_bins, s->d_del.as<int32_t>(),
                                              s->d_gsz.as<int64_t>(), st);
        // one copy back: {candidate, group size, index} a group
        std::vector<DelegateD> h((size_t)ng);
        ScratchBuf recs;
        recs.ensure(sizeof(DelegateD) * (size_t)ng);
        launch_pack_delegates(s->heap.as<CandD>(), s->d_del.as<int32_t>(), s->d_gsz.as<int64_t>(), ng,
                              recs.as<DelegateD>(), st);
        SPS_HIP(hipMemcpyAsync(h.data(), recs.p, sizeof(DelegateD) * (size_t)ng, hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        recs.idle();
        s->h_del.reserve((size_t)ng);
        s->h_gsz.reserve((size_t)ng);
        s->h_del_cand.reserve((size_t)ng);
        for (const DelegateD& d : h) {
            s->h_del.push_back(d.index);
            s->h_gsz.push_back(d.size);
            s->h_del_cand.push_back({d.c.mt, d.c.mdt, d.c.mwidth, d.c.msnr});
        }
        *h_ngroups = ng;
    });
}

SPS_API sps_status sps_search_get_delegates(const sps_search* s, sps_cand* h_delegates, int64_t* h_group_sizes,
                                            int64_t cap, int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(s && h_n && cap >= 0, "null argument");
        const int64_t ng = (int64_t)s->h_del.size();
        *h_n = ng;
        const int64_t m = std::min(ng, cap);
        for (int64_t i = 0; i < m; ++i) {
            if (h_delegates) h_delegates[i] = s->h_del_cand[(size_t)i];
            if (h_group_sizes) h_group_sizes[i] = s->h_gsz[(size_t)i];
        }
    });
}

SPS_API sps_status sps_search_write_log(const sps_search* s, const char* filename, float delt_bin,
                                        float t_chunk_begin) {
    if (!s || !filename) {
        g_last_error = "null argument";
        return SPS_ERR_INVALID_ARGUMENT;
    }
    return sps_write_log(reinterpret_cast<const sps_cand*>(s->heap.p), s->heap_n, s->h_del.data(), s->h_gsz.data(),
                         (int64_t)s->h_del.size(), filename, delt_bin, t_chunk_begin);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// batched multi-beam search
//
// Every beam is a full search (its own plan, tables and statistics).  Beams
// are spread over a few worker streams by longest-first greedy assignment on
// their byte cost; the beams of one worker run one after the other and share
// one set of scratch buffers sized for the largest of them, so the HBM held
// is the inputs, the candidate buffers and nworkers x the largest beam's
// states.  The whole fork/join launch sequence is captured once into a HIP
// graph and replayed; it holds kernels and event waits only.
// ---------------------------------------------------------------------------
struct sps_batch {
    struct Beam {
        sps_batch_beam io{};
        std::unique_ptr<sps_search> s;
        int worker = 0;
        double cost = 0.0;
    };
    struct Worker {
        hipStream_t st = nullptr;
        hipEvent_t join = nullptr;
        DevBuf sa, sb, na, nb, nimg, dmt;
        sps_search::Scratch sc;
        std::vector<int64_t> beams;
    };
    sps_batch_params p{};
    std::vector<Beam> beams;
    std::vector<Worker> workers;
    hipEvent_t fork = nullptr;
    hipStream_t cap = nullptr;  // capture origin
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool prepared = false;

    ~sps_batch() {
        drop_graph();
        for (auto& w : workers) {
            if (w.join) (void)hipEventDestroy(w.join);
            if (w.st) (void)hipStreamDestroy(w.st);
        }
        if (fork) (void)hipEventDestroy(fork);
        if (cap) (void)hipStreamDestroy(cap);
    }

    void drop_graph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }

    void assign() {
        std::vector<int64_t> order(beams.size());
        for (size_t i = 0; i < order.size(); ++i) order[i] = (int64_t)i;
        std::stable_sort(order.begin(), order.end(),
                         [&](int64_t a, int64_t b) { return beams[(size_t)a].cost > beams[(size_t)b].cost; });
        std::vector<double> load(workers.size(), 0.0);
        for (auto& w : workers) w.beams.clear();
        for (int64_t b : order) {
            const size_t w = (size_t)(std::min_element(load.begin(), load.end()) - load.begin());
            load[w] += beams[(size_t)b].cost;
            beams[(size_t)b].worker = (int)w;
        }
        // each worker runs its beams in index order
        for (size_t b = 0; b < beams.size(); ++b) workers[(size_t)beams[b].worker].beams.push_back((int64_t)b);
    }

    void prepare(hipStream_t st) {
        if (prepared) return;
        for (auto& b : beams) {
            b.s->setup(st, false);
            // (no allocation while the beams are captured)
            const int64_t N = b.s->p.nsamps;
            if (b.io.d_dmt)
                if (const size_t n = b.s->f->overlap_bytes(b.io.d_in, p.in_dtype == SPS_U8, N, N, b.io.d_dmt, N))
                    b.s->f->in_copy.ensure(n);
        }
        for (auto& w : workers) {
            sps_search::ScratchSize m;
            bool need_dmt = false;
            for (int64_t b : w.beams) {
                const auto z = beams[(size_t)b].s->scratch_size();
                m.sa = std::max(m.sa, z.sa);
                m.sb = std::max(m.sb, z.sb);
                m.na = std::max(m.na, z.na);
                m.nb = std::max(m.nb, z.nb);
                m.nimg = std::max(m.nimg, z.nimg);
                if (!beams[(size_t)b].io.d_dmt) {
                    m.dmt = std::max(m.dmt, z.dmt);
                    need_dmt = true;
                }
            }
            if (w.beams.empty()) continue;
            w.sa.ensure(sizeof(float) * (size_t)m.sa);
            w.sb.ensure(sizeof(float) * (size_t)m.sb);
            if (p.snr_norm) {
                w.na.ensure(sizeof(float) * (size_t)m.na);
                w.nb.ensure(sizeof(float) * (size_t)m.nb);
                w.nimg.ensure(sizeof(float) * (size_t)m.nimg);
            }
            if (need_dmt) w.dmt.ensure(sizeof(float) * (size_t)m.dmt);
            w.sc.sa = w.sa.as<float>();
            w.sc.sb = w.sb.as<float>();
            w.sc.na = w.na.as<float>();
            w.sc.nb = w.nb.as<float>();
            w.sc.nimg = w.nimg.as<float>();
            w.sc.dmt = w.dmt.as<float>();
        }
        SPS_HIP(hipStreamSynchronize(st));
        prepared = true;
    }

    // fork on `origin`, every worker runs its beams, join back on `origin`
    void enqueue(hipStream_t origin) {
        SPS_HIP(hipEventRecord(fork, origin));
        for (auto& w : workers) {
            if (w.beams.empty()) continue;
            SPS_HIP(hipStreamWaitEvent(w.st, fork, 0));
            for (int64_t bi : w.beams) {
                Beam& b = beams[(size_t)bi];
                b.s->enqueue(b.io.d_in, b.io.d_dmt, b.io.d_cands, b.io.d_count, w.st, w.sc, nullptr);
            }
            SPS_HIP(hipEventRecord(w.join, w.st));
            SPS_HIP(hipStreamWaitEvent(origin, w.join, 0));
        }
    }

    void capture() {
        drop_graph();
        SPS_HIP(hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal));
        try {
            enqueue(cap);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(cap, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        SPS_HIP(hipStreamEndCapture(cap, &graph));
        SPS_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    }
};

extern "C" {

SPS_API sps_status sps_batch_create(const sps_batch_params* p, const sps_batch_beam* beams, int64_t nbeams,
                                    sps_batch** out) {
    return guarded([&] {
        SPS_REQUIRE(p && out && (nbeams == 0 || beams), "null argument");
        *out = nullptr;
        SPS_REQUIRE(nbeams >= 1, "a batch needs at least one beam");
        SPS_REQUIRE(p->nworkers >= 1 && p->nworkers <= 8, "nworkers must be 1..8");
        std::unique_ptr<sps_batch> b(new sps_batch());
        b->p = *p;
        b->beams.resize((size_t)nbeams);
        for (int64_t i = 0; i < nbeams; ++i) {
            const sps_batch_beam& io = beams[i];
            SPS_REQUIRE(io.d_in && io.d_count, "null beam buffer");
            SPS_REQUIRE(io.cand_capacity >= 0 && (io.cand_capacity == 0 || io.d_cands), "bad candidate buffer");
            sps_search_params sp{};
            sp.f_min = io.f_min;
            sp.f_max = io.f_max;
            sp.tsamp = io.tsamp;
            sp.nchans = io.nchans;
            sp.nsamps = io.nsamps;
            sp.dt_max = io.dt_max;
            sp.in_dtype = p->in_dtype;
            sp.norm_mode = p->norm_mode;
            sp.snr_norm = p->snr_norm;
            sp.box_q = p->box_q;
            sp.threshold = p->threshold;
            sp.cand_capacity = io.cand_capacity;
            sps_batch::Beam& bm = b->beams[(size_t)i];
            bm.io = io;
            bm.s = make_search(&sp);
            // byte cost of the beam: input read twice, every state written
            // once and read once, the image read by the boxcar
            const EnginePlan& e = bm.s->f->eng;
            double rows = (double)e.nchans * 2.0 + (double)e.rows[0];
            for (int k = 1; k <= e.niters; ++k) rows += (double)(e.rows[(size_t)k - 1] + e.rows[(size_t)k]);
            bm.cost = rows * (double)e.nsamps;
        }
        b->workers = std::vector<sps_batch::Worker>((size_t)std::min<int64_t>(p->nworkers, nbeams));
        for (auto& w : b->workers) {
            SPS_HIP(hipStreamCreateWithFlags(&w.st, hipStreamNonBlocking));
            SPS_HIP(hipEventCreateWithFlags(&w.join, hipEventDisableTiming));
        }
        SPS_HIP(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
        SPS_HIP(hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking));
        b->assign();
        *out = b.release();
    });
}

SPS_API sps_status sps_batch_destroy(sps_batch* b) {
    return guarded([&] {
        delete b;
        scratch_trim();
    });
}

SPS_API sps_status sps_batch_get_beam_info(const sps_batch* b, int64_t beam, int64_t* h_ndt, int32_t* h_worker,
                                           int64_t* h_niters) {
    return guarded([&] {
        SPS_REQUIRE(b, "null handle");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        const auto& bm = b->beams[(size_t)beam];
        if (h_ndt) *h_ndt = bm.s->ndt;
        if (h_worker) *h_worker = bm.worker;
        if (h_niters) *h_niters = bm.s->f->eng.niters;
    });
}

SPS_API sps_status sps_batch_set_schedule(sps_batch* b, int64_t beam, const int32_t* h_depths, int64_t n) {
    return guarded([&] {
        SPS_REQUIRE(b && (n == 0 || h_depths), "null argument");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        b->beams[(size_t)beam].s->f->set_schedule(std::vector<int>(h_depths, h_depths + n));
        b->drop_graph();
        b->prepared = false;  // the new pass tables are built before the next capture
    });
}

SPS_API sps_status sps_batch_set_group_shape(sps_batch* b, int64_t beam, int lds_floats, int max_rows, int tiles_per_block) {
    return guarded([&] {
        SPS_REQUIRE(b, "null handle");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        b->beams[(size_t)beam].s->f->set_group_shape(lds_floats, max_rows, tiles_per_block);
        b->drop_graph();
        b->prepared = false;
    });
}

SPS_API sps_status sps_batch_set_staged(sps_batch* b, int64_t beam, int staged) {
    return guarded([&] {
        SPS_REQUIRE(b, "null handle");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        b->beams[(size_t)beam].s->f->set_staged(staged);
        b->drop_graph();
        b->prepared = false;
    });
}

SPS_API sps_status sps_batch_get_schedule(const sps_batch* b, int64_t beam, int32_t* h_depths, int64_t cap,
                                          int64_t* h_n) {
    return guarded([&] {
        SPS_REQUIRE(b && h_n, "null argument");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        const auto& s = b->beams[(size_t)beam].s->f->schedule;
        *h_n = (int64_t)s.size();
        for (int64_t i = 0; i < *h_n && i < cap && h_depths; ++i) h_depths[i] = s[(size_t)i];
    });
}

SPS_API sps_status sps_batch_run(sps_batch* b, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(b, "null handle");
        hipStream_t st = as_stream(stream);
        b->prepare(st);
        b->enqueue(st);
    });
}

SPS_API sps_status sps_batch_launch(sps_batch* b, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(b, "null handle");
        hipStream_t st = as_stream(stream);
        b->prepare(st);
        if (!b->exec) b->capture();
        SPS_HIP(hipGraphLaunch(b->exec, st));
    });
}

SPS_API sps_status sps_batch_sort_candidates(sps_batch* b, int64_t beam, int64_t* h_count, void* stream) {
    return guarded([&] {
        SPS_REQUIRE(b && h_count, "null argument");
        SPS_REQUIRE(beam >= 0 && beam < (int64_t)b->beams.size(), "beam index out of range");
        auto& bm = b->beams[(size_t)beam];
        hipStream_t st = as_stream(stream);
        unsigned long long n = 0;
        SPS_HIP(hipMemcpyAsync(&n, bm.io.d_count, sizeof(n), hipMemcpyDeviceToHost, st));
        SPS_HIP(hipStreamSynchronize(st));
        const int64_t m = std::min<int64_t>((int64_t)n, bm.io.cand_capacity);
        sort_cands(reinterpret_cast<CandD*>(bm.io.d_cands), m, bm.s->ndt, bm.s->p.nsamps, bm.s->p.box_q, st);
        *h_count = (int64_t)n;
        if ((int64_t)n > bm.io.cand_capacity)
            throw Error(SPS_ERR_CAPACITY, "more candidates than the beam's cand_capacity");
    });
}

}  // extern "C"
