// launch_limits.hpp -- how much one launch's grid takes.
#pragma once

#include <cstdint>

namespace sps {

// A dispatch counts its threads in 32 bits per dimension, and HIP refuses a
// grid with more, whatever its number of blocks.
constexpr int64_t kMaxGridThreads = 0xffffffffLL;

// Rows of a launch that gives each row `blocks` blocks of `threads` threads in
// one dimension (0: not even one).
constexpr int64_t rows_per_launch(int64_t blocks, int64_t threads) { return kMaxGridThreads / (blocks * threads); }

}  // namespace sps
