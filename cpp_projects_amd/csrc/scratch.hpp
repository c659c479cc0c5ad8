// scratch.hpp -- device scratch of the calls that synchronise before they
// return.  hipMalloc and hipFree of such a call's buffers cost 20 to 300 us
// each and hipFree waits for the device, so blocks go to a small process-wide
// list of idle ones instead.
#pragma once

#include <cstddef>
#include <cstdint>

#include "common.hpp"

namespace sps {

// One block of device memory.  Its user calls idle() once the stream that used
// it has been synchronised; only then is the block kept for another call
// (whatever thread or stream that is), otherwise it is freed.
class ScratchBuf {
public:
    ScratchBuf() = default;
    ScratchBuf(const ScratchBuf&) = delete;
    ScratchBuf& operator=(const ScratchBuf&) = delete;
    ~ScratchBuf() { release(); }
    // at least n bytes, contents lost (an older block only after a synchronisation)
    void ensure(size_t n);
    void idle() { idle_ = true; }
    template <class T>
    T* as() const {
        return static_cast<T*>(p);
    }

    void* p = nullptr;
    size_t bytes = 0;

private:
    void release();
    int device_ = 0;
    bool idle_ = false;
};

// One block cut into 256-byte aligned pieces.
class Arena {
public:
    template <class T>
    size_t add(int64_t n) {
        const size_t at = bytes_;
        bytes_ += (sizeof(T) * (size_t)(n > 1 ? n : 1) + 255) / 256 * 256;
        return at;
    }
    void allocate() { buf_.ensure(bytes_); }
    void idle() { buf_.idle(); }
    template <class T>
    T* at(size_t off) const {
        return reinterpret_cast<T*>(buf_.as<uint8_t>() + off);
    }

private:
    size_t bytes_ = 0;
    ScratchBuf buf_;
};

}  // namespace sps
