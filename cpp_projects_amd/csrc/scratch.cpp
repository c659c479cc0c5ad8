// scratch.cpp -- the list of idle scratch blocks (scratch.hpp).
#include "scratch.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace sps {

namespace {

// What is kept at most, all devices together: enough for the sort of some ten
// million candidates.  Larger blocks are freed as they come back, the whole
// list when a handle is destroyed, an allocation fails or a caller asks for it.
constexpr size_t kKeepBytes = (size_t)256 << 20;
constexpr size_t kKeepBlocks = 16;
// Requests below this take no block above it, so that a counter does not hold
// the block that the next sort needs; a larger one takes the smallest that fits,
// and a gather finds more room in it.
constexpr size_t kSmall = (size_t)1 << 20;

struct Block {
    void* p;
    size_t bytes;
    int device;
};

struct Idle {
    std::mutex m;
    std::vector<Block> blocks;  // oldest first
    size_t bytes = 0;
};

// never destroyed: other statics' destructors may still call the library
Idle& idle_list() {
    static Idle* l = new Idle();
    return *l;
}

// sizes in eighths of a power of two, so that calls of similar size share blocks
size_t block_size(size_t n) {
    size_t g = (size_t)64 << 10;
    while (g * 16 <= n) g *= 2;
    return (n + g - 1) / g * g;
}

}  // namespace

void scratch_trim() noexcept {
    std::vector<Block> old;
    {
        Idle& l = idle_list();
        std::lock_guard<std::mutex> lock(l.m);
        old.swap(l.blocks);
        l.bytes = 0;
    }
    for (const Block& b : old) (void)hipFree(b.p);
}

void ScratchBuf::ensure(size_t n) {
    if (p && n <= bytes) return;
    idle_ = idle_ || p;  // (a caller that grows a block has synchronised)
    release();
    n = block_size(n);
    SPS_HIP(hipGetDevice(&device_));
    {
        Idle& l = idle_list();
        std::lock_guard<std::mutex> lock(l.m);
        size_t best = l.blocks.size();
        for (size_t i = 0; i < l.blocks.size(); ++i)
            if (l.blocks[i].device == device_ && l.blocks[i].bytes >= n && (n >= kSmall || l.blocks[i].bytes <= kSmall) &&
                (best == l.blocks.size() || l.blocks[i].bytes < l.blocks[best].bytes))
                best = i;
        if (best < l.blocks.size()) {
            p = l.blocks[best].p;
            bytes = l.blocks[best].bytes;
            l.bytes -= bytes;
            l.blocks.erase(l.blocks.begin() + (long)best);
        }
    }
    if (!p) {
        device_malloc(&p, n);
        bytes = n;
    }
}

void ScratchBuf::release() {
    if (!p) return;
    Block b{p, bytes, device_};
    const bool keep = idle_ && b.bytes <= kKeepBytes;
    p = nullptr;
    bytes = 0;
    idle_ = false;
    std::vector<Block> out;
    if (keep) {
        Idle& l = idle_list();
        std::lock_guard<std::mutex> lock(l.m);
        try {
            l.blocks.reserve(kKeepBlocks + 1);
            out.reserve(kKeepBlocks + 1);
        } catch (...) {
            (void)hipFree(b.p);
            return;
        }
        l.blocks.push_back(b);
        l.bytes += b.bytes;
        while (l.bytes > kKeepBytes || l.blocks.size() > kKeepBlocks) {
            out.push_back(l.blocks.front());
            l.bytes -= l.blocks.front().bytes;
            l.blocks.erase(l.blocks.begin());
        }
    }
    if (!keep) (void)hipFree(b.p);
    for (const Block& o : out) (void)hipFree(o.p);
}

}  // namespace sps
