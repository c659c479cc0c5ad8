// stack_plan.hpp -- host tables of the stacked merge passes.
//
// A stacked pass runs up to six merge iterations in one launch, in two stages
// through LDS: a block owns a group of consecutive output rows and a time
// tile, stages the distinct rows of the pass's input state that the group's
// trees read (the leaves), evaluates the rows of an intermediate state from
// them into LDS (stage A, up to three iterations), and the group's output rows
// from those (stage B, up to three more).  An intermediate row is shared by
// every output row that reads it, so six iterations cost two depth-3 trees
// per output instead of a depth-6 one.
//
// Every row in LDS is a window of times: read with shifts smin..smax, it holds
// [T - smax, T + tile - smin).  Times below 0 hold -0.0f, and so does a
// reserved zero window that a missing head (a copied row) points to: x + -0.0f
// is x for every x, so neither case needs a branch.
#pragma once

#include <cstdint>
#include <vector>

#include "plan.hpp"

namespace sps {

constexpr int kStackTile = 128;     // samples per tile
constexpr int kStackThreads = 1024;  // threads per block
constexpr int kStackSlots = 4;      // 4-sample units (leaf windows) per thread
constexpr int kStackMaxUnits = kStackThreads * kStackSlots;
constexpr int kStackMaxDepth = 6;   // iterations per pass: two stages of at most three
constexpr int64_t kStackMaxSamps = (int64_t)1 << 30;  // times are 32-bit in the kernel
constexpr int kStackMaxLeaves = 255;  // leaf indices of the unit table are bytes
constexpr int kStackMaxChans = 128;   // channels of a group that builds state 0
// LDS of a block (floats): two blocks per CU of 160 KiB with what is static
constexpr int kStackLdsFloats = 19200;
// packed lanes of an intermediate row's samples before its last `tile` ones
constexpr int kStackTailLanes = 8;

// A slot of a pass that builds state 0: the unit's channel and that channel's
// place in its group, in one register.
constexpr int kStackChanBits = 25;
static_assert(kStackMaxChans <= 1 << (32 - kStackChanBits), "places fit above the channel");
constexpr uint32_t stack_slot(uint32_t chan, uint32_t place) { return chan | place << kStackChanBits; }
constexpr uint32_t slot_chan(uint32_t s) { return s & ((1u << kStackChanBits) - 1); }
constexpr uint32_t slot_place(uint32_t s) { return s >> kStackChanBits; }

// One row of a stage, 32 bytes (one scalar load): its value at the window's
// main sample i (the last `tile` of them) is the tree over the floats at LDS
// places c_j + i, j < 2^L, in heap-leaf order.  L <= 2: w[j] is the byte offset
// of c_j; L = 3: w[j / 2] holds the float offsets of c_j (low half, even j) and
// of the next.  Stage A writes LDS bytes out + 4 i; stage B output row `out`
// at T + i.
struct StackRow {
    uint32_t w[4];
    int32_t out;
    int32_t pad[3];
};
// Rows past the end that a wave may load ahead (and not use).
constexpr int kStackRowPad = kStackThreads / 64;
// Up to kStackTailLanes samples of a stage-A row before its main samples
// (c: byte offsets).
struct StackTail {
    int32_t c[8];
    int32_t out;
    int32_t n;
    int32_t pad[2];  // 48 bytes: copied to LDS 16 at a time
};
// A leaf row of the input state: 4-sample units over [T - smax4, ...).
struct StackLeaf {
    int64_t row;      // state row (or channel, when the pass builds state 0)
    int32_t smax4;    // a multiple of 4
    int32_t lds_off;  // float offset of its window (a multiple of 4)
    int32_t nunits;
    int32_t unit0;    // its first unit in the group's numbering
};
// An init row k >= 1 of a channel, built in LDS from the channel's row 0:
// sample q (time T - t_off + q) reads row 0 at lds[c + q - j], j <= k.
struct StackInitRow {
    int32_t c;
    int32_t k;
    int32_t out;
    int32_t n;      // samples of its window
    int32_t t_off;  // smax of its window
    int32_t pad[3];
};
struct StackGroup {
    int64_t unit0;  // first entry of the group in the unit -> leaf table
    int32_t leaf0, nleaves, nunits;
    int32_t init0, ninit;
    int32_t row_a0, nrows_a;
    int32_t tail0, ntails;
    int32_t row_b0, nrows_b;
    int32_t zero_off;  // float offset of the zero window (kStackTile floats)
    int32_t tail_off;  // float offset of the copy of the group's tails (a multiple of 4)
    int32_t smax4;     // largest smax4 of its leaves
};

struct StackTables {
    int la = 0, lb = 0;  // iterations of stages A and B (0: it copies)
    bool init = false;   // leaves are channels: the pass builds state 0 itself
    int lds_floats = 0;  // dynamic LDS of a block
    std::vector<StackGroup> groups;
    std::vector<StackLeaf> leaves;
    std::vector<uint8_t> unit_leaf;
    std::vector<StackInitRow> inits;
    std::vector<StackRow> rows_a, rows_b;
    std::vector<StackTail> tails;
};

// The tables of the pass over iterations i0 .. i0 + depth - 1 of a plan whose
// live rows (per state) are flagged in `live`.  init: the pass reads the
// waterfall and builds its state-0 leaves (i0 == 1; init dts 0 .. K-1 per
// channel).  Throws std::runtime_error when a single output row does not fit, or
// (init) a channel does not fit stack_slot.
//
// weigh_init: gives up (returns no tables, `init` false) where state 0 should be
// left to a launch of its own.  Every group builds the init rows that it reads
// anew, row k in k steps from row 0, and their windows take LDS from its
// outputs, so a group has fewer of them and more groups build the same row.
// Above two steps per output sample that is slower than a state 0 in memory (64
// channels x 131072, us in the pass and before it: dt 512, 11.1 steps, 1102 and
// 176; dt 192, 2.1, 135 and 90; dt 128, 0.9, 68 and 74), once the steps of the
// launch pass 16 M: with fewer, the second launch and the few blocks of the
// separate init cost more (dt 384: 48 x 12000, 12 M steps, 35 and 52; 64 x 6000,
// 18 M, 47 and 38).
StackTables build_stack_pass(const EnginePlan& eng, const std::vector<std::vector<uint8_t>>& live, int i0, int depth,
                             bool init, bool weigh_init = false);

// Threads of a block for these tables: 1024, or 256 and 128 where no group has
// more than 16 and 4 rows in a stage and their slots hold its units.  A plan of
// few channels has one such group; most of 16 waves then wait for the few with a
// row, tile after tile, where a CU can hold 8 and 16 small blocks (us at 4 M
// samples with 1024, 256 and 128 threads: 2 channels of 3 rows 108, 42, 31; 4 of
// 13 rows 159, 87, 83, and at 200000 samples 16.9, 11.8, 15.2).
constexpr int kStackFew16 = 256, kStackFew4 = 128;
int stack_threads(const StackTables& t);

}  // namespace sps
