// kernels.hpp -- host launchers for the gfx950 kernels (defined in *.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sps {

// init formulas as seen by the kernels (same values as sps_init_mode)
constexpr int kInitMeanD = 0;
constexpr int kInitRestrictD = 1;
constexpr int kInitCFdmtD = 2;

// One merge output row: out[t] = tail[t] + (t >= offset ? head[t - offset] : 0),
// or a verbatim copy of tail when head < 0.
struct RowDescD {
    int64_t out_row;
    int64_t tail_row;
    int64_t head_row;
    int64_t offset;
};

// Per-channel normalisation applied while the FDMT init reads the waterfall:
// v = keep ? (x - mu) / sigma : 0 (or keep ? 1 : 0 for the mask transform).
struct ChanNorm {
    const float* mu;       // per channel
    const float* sigma;    // per channel
    const uint8_t* keep;   // per channel
};

// FDMT init: rows of state 0 for every channel.
//   in: nchans x nsamps (f32 or u8; ignored when ones), in_pitch elements
//   norm: nullptr, or per-channel normalisation
//   d_live: nullptr, or per state-0 row flags; rows flagged 0 are not stored
//   grid_consec: every channel's init dts are 0, 1, ..., K-1 with K <= 5
//     (enables the register fast path of the mean init)
void launch_fdmt_init(int mode, const void* in, int in_u8, int ones, int64_t in_pitch, const ChanNorm* norm,
                      int64_t nchans, int64_t nsamps, const int32_t* d_grid, const int64_t* d_grid_off,
                      const int64_t* d_chan_row_off, float* state, int64_t pitch, hipStream_t st,
                      int dmax_all = -1,  // largest init dt of any channel; < 0 selects the unstaged kernel
                      const uint8_t* d_live = nullptr, int grid_consec = 0);

// Optional epilogue of the last merge: divide by sqrtf(n + 1e-8) with n from
// nrm (rows x nrm_len) for t < nrm_len and stats[4] (kept channels) beyond.
struct MergeEpilogue {
    const float* nrm;
    int64_t nrm_len;
    const double* stats;
};

// One merge iteration over nrows descriptors; rows with out_row >= out_rows_limit are skipped.
void launch_fdmt_merge(const float* in, int64_t in_pitch, float* out, int64_t out_pitch, const RowDescD* d_rows,
                       int64_t nrows, int64_t nsamps, int64_t out_rows_limit, hipStream_t st,
                       const MergeEpilogue* snr = nullptr);

// Stacked pass (stack_plan.hpp): its tables on the device.
struct StackPassDev {
    const void* groups = nullptr;
    const void* leaves = nullptr;
    const uint8_t* unit_leaf = nullptr;
    const void* inits = nullptr;
    const void* rows_a = nullptr;
    const void* rows_b = nullptr;
    const void* tails = nullptr;
    int64_t ngroups = 0;
    int la = 0, lb = 0, lds_floats = 0, threads = 0;
    bool init = false;
};
// Sets what the stacked kernels need (their LDS above 64 KiB); called on the
// current device before their first launch.
void prepare_stack_kernels();
// kind 0: in is a state (16-byte aligned, in_pitch % 4 == 0); 1, 2, 3: an f32
// or u8 waterfall (any alignment and pitch) or ones, from which the pass
// builds state 0 (norm: optional per-channel normalisation; plain_row0: row 0
// is the sample itself rather than 0 + the sample).
void launch_stack_pass(const StackPassDev& p, int kind, const void* in, int64_t in_pitch, const ChanNorm* norm,
                       bool plain_row0, float* out, int64_t out_pitch, int64_t nsamps, hipStream_t st,
                       const MergeEpilogue* snr = nullptr);

// Adjoint of `depth` merges (1..kAdjMaxDepth): g_prev[p][t] is the sum over row
// p's users of g_out[row][t + shift] (t + shift < nsamps), nested as one
// iteration after the other adds.  A user is a row of the source state that row
// p feeds; closes = how many of the sums in between (innermost first) end with
// it.  d_off: each row's range of d_users.
struct AdjUser {
    int64_t shift;
    uint32_t row, closes;
};
void launch_fdmt_merge_adjoint(const float* g_out, int64_t out_pitch, float* g_prev, int64_t prev_pitch, int depth,
                               const int64_t* d_off, const AdjUser* d_users, int64_t prev_rows, int64_t nsamps,
                               hipStream_t st);

// Adjoint of the (mean) init: g_x[c][i] = sum_k sum_{t=max(i,d_k)}^{min(i+d_k,N-1)} g_s[k][t] / (d_k+1).
// dmax: the largest d of any channel.
void launch_fdmt_init_adjoint(const float* g_state, int64_t pitch, float* g_x, int64_t x_pitch, int64_t nchans,
                              int64_t nsamps, const int32_t* d_grid, const int64_t* d_grid_off,
                              const int64_t* d_chan_row_off, int dmax, hipStream_t st);

// ---- statistics / normalisation ----
// row sums in FP64 (fixed lane partition) -> row mean / variance (double)
void launch_row_stats(const void* in, int in_u8, int64_t rows, int64_t cols, double* d_row_mean, double* d_row_var,
                      hipStream_t st);
// global stats + keep flags + per-channel (mu, sigma) floats; d_stats (6 doubles):
// mean, std, var_mean, var_std, n_keep, unused; d_buff (optional) gets the
// reference float layout {means[R], vars[R], mean, std, var_mean, var_std}
void launch_stats_finalize(const double* d_row_mean, const double* d_row_var, int64_t rows, int mode,
                           double* d_stats, float* d_mu, float* d_sigma, uint8_t* d_keep, float* d_buff,
                           hipStream_t st,
                           unsigned long long* d_clear = nullptr);
void launch_apply_norm(float* x, float* mask, int64_t rows, int64_t cols, const float* d_mu, const float* d_sigma,
                       const uint8_t* d_keep, hipStream_t st);
void launch_fdmt_normalization(const float* a, const float* n, int64_t len, float* out, hipStream_t st);
void launch_fdmt_normalization_rows(const float* a, int64_t rows, int64_t cols, const float* n, int64_t norm_cols,
                                    float* out, hipStream_t st);
// S/N normalisation of the DM-time image by the mask transform: for t < norm_len
// the divisor comes from d_norm (rows x norm_len), beyond it from *d_nkeep.
// The transform of a row-constant 0/1 keep mask over its first L columns,
// counted: out[r][t] = #{c : keep[c], shift[r][c] <= t} (shift: the
// accumulated delay of channel c in output row r, an int16 table; L <= 16000)
void launch_mask_counts(const int16_t* shift, const uint8_t* keep, int64_t rows, int64_t nchans, int L, float* out,
                        int64_t pitch, hipStream_t st);
void launch_snr_normalise(float* img, int64_t rows, int64_t cols, int64_t pitch, const float* d_norm,
                          int64_t norm_len, const double* d_stats, hipStream_t st);

// ---- boxcar ----
struct CandD {
    int32_t mt, mdt, mwidth;
    float msnr;
};
// Emits every (row, t, width) with window sum / sqrtf(w) > *d_thr (strict), unordered.
// pow2: widths 1,2,..,wmax (wmax a power of two), mwidth = log2 w; else widths 1..wmax, mwidth = w.
void launch_boxcar(const float* img, int64_t rows, int64_t cols, int64_t pitch, const float* d_thr, float h_thr,
                   int wmax, int pow2, CandD* out, int64_t cap, unsigned long long* d_count, hipStream_t st);
void launch_boxcar_snr(const float* img, int64_t rows, int64_t cols, int w, float* snr, hipStream_t st);
void launch_boxcar_snr_adjoint(const float* g, int64_t rows, int64_t cols, int w, float* gi, hipStream_t st);
// x[i] = floorf(x[i]) for i < n
void launch_digitize(float* x, int64_t n, hipStream_t st);
void launch_detect_max(const float* a, const float* n, int64_t rows, int64_t cols, int wnd, void* d_block_best,
                       int64_t nblocks_cap, void* d_out, hipStream_t st);
int64_t detect_max_blocks(int64_t rows, int64_t cols);
// tiled detectors of the reference's per-block kernels (mode 1: boxcar S/N of
// x / sqrtf(1e-7 + n) inside a tile; mode 2: energy ratio sqrt(sum x^2 / sum n^2));
// per-tile results in the caller's arrays of rows * ceil(cols / tile) entries
void launch_detect_tiles(int mode, const float* x, const float* n, int64_t rows, int64_t cols, int tile, int wnd,
                         float* tile_val, int32_t* tile_pos, int32_t* tile_w, void* d_out, hipStream_t st);
// zeroes the rows not kept, writes a byte mask and {row variances, mean, std of variances}
void launch_clean_rows(float* x, uint8_t* mask, int64_t rows, int64_t cols, const uint8_t* d_keep,
                       const double* d_row_var, const double* d_stats, float* d_buff, hipStream_t st);

// ---- sorting / scans / clustering ----
// stable LSD radix sort of (key, val) pairs over key bits [0, nbits) (K:
// uint32_t or uint64_t); tmp buffers of n entries each, scratch of
// sort_scratch_bytes(n) that the launch which makes the n keys clears (the
// launch_*_keys below).  True: the result is in the tmp buffers.
template <typename K>
bool radix_sort_pairs(K* keys, uint32_t* vals, K* keys_tmp, uint32_t* vals_tmp, int64_t n, int nbits, void* scratch,
                      hipStream_t st);
size_t sort_scratch_bytes(int64_t n);
// inclusive scan of n uint32 values in place; scratch of scan_scratch_entries(n)
void scan_inclusive_u32(uint32_t* data, int64_t n, uint32_t* scratch, hipStream_t st);
// the same for floats: per-thread sums of 4 in order, a block tree over them,
// block prefixes added last (deterministic, not the sequential order)
void scan_inclusive_f32(float* data, int64_t n, float* scratch, hipStream_t st);
int64_t scan_scratch_entries(int64_t n);

template <typename K>
void launch_cand_keys(const CandD* c, int64_t n, int bits_t, int bits_w, K* keys, uint32_t* vals, void* scratch,
                      hipStream_t st);
template <typename K>
void launch_cand_from_keys(const K* keys, const uint32_t* vals, int64_t n, int bits_t, int bits_w, CandD* out,
                           hipStream_t st);
// {smallest, largest} of each member (mt, mdt, mwidth) as ordered uint32
// (value ^ 0x80000000), into six words that hold {0xffffffff, 0} three times
void launch_cand_ranges(const CandD* c, int64_t n, uint32_t* ranges, hipStream_t st);
// keys (group << bits | member - base) and vals of one clustering level, in
// the order perm (null: the candidates' own, one group)
template <typename K>
void launch_cluster_keys(const CandD* c, const uint32_t* perm, const uint32_t* group, int64_t n, int member,
                         uint32_t base, int bits, K* keys, uint32_t* vals, void* scratch, hipStream_t st);
// all three levels in one launch where n is small enough (false: it is not):
// the permutation, group starts and ids, {smallest, largest ord(mt), groups}
bool launch_cluster_small(const CandD* c, int64_t n, const int32_t* d_bins, uint32_t* perm, uint32_t* flags,
                          uint32_t* group, uint32_t* info, hipStream_t st);
// group starts and 1-based group ids of sorted keys (scratch as for the sort)
template <typename K>
void launch_cluster_groups(const K* keys, int64_t n, int bits, const int32_t* d_bins, int level, void* scratch,
                           uint32_t* flags, uint32_t* group, hipStream_t st);
void launch_cluster_delegates(const CandD* c, const uint32_t* perm, const uint32_t* gid, const uint32_t* flags,
                              int64_t n, unsigned long long* best, uint32_t* start, hipStream_t st);
void launch_delegate_keys(const CandD* c, const unsigned long long* best, int64_t ng, uint32_t base, uint32_t* keys,
                          uint32_t* vals, void* scratch, hipStream_t st);
void launch_delegate_out(const unsigned long long* best, const uint32_t* start, const uint32_t* order, int64_t ng,
                         int64_t n, int32_t* delegates, int64_t* sizes, hipStream_t st);
// per caller group [begin[g], begin[g+1]) of idx: the index with the largest msnr (first on ties)
void launch_select_delegates(const CandD* c, const int32_t* idx, int64_t nidx, const int32_t* begin, int64_t ngroups,
                             int32_t* out, hipStream_t st);
// 8-bit raw voltages -> overlapping complex FFT blocks out[pol][fft][chan][bin]
// (re/im float pairs; GUPPI input [chan][samp][npol], LOFAR [npol][samp][chan])
void launch_unpack_guppi(const int8_t* in, int64_t nsamp, int noverlap, int nbin, int nfft, int npol, int nchan,
                         float* out, hipStream_t st);
void launch_unpack_lofar(const int8_t* in, int64_t nsamp, int noverlap, int nbin, int nfft, int npol, int nchan,
                         float* out, hipStream_t st);
// a group's delegate, as it is read back
struct DelegateD {
    CandD c;
    int64_t size;
    int32_t index, pad;
};
void launch_pack_delegates(const CandD* c, const int32_t* del, const int64_t* size, int64_t ng, DelegateD* out,
                           hipStream_t st);
void launch_fill_u64(unsigned long long* v, int64_t n, unsigned long long val, hipStream_t st);

}  // namespace sps
