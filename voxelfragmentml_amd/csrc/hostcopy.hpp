// Copies of device memory to a caller's host memory.
#pragma once
#include <memory>
#include <thread>
#include <vector>

#include "common.hpp"

namespace vf {

// Between two looks at a word that the device or another thread will change: a few pauses of the core, for waits of a
// microsecond or two, then the core goes to any other thread that wants it.
class HostPause {
public:
    void operator()()
    {
        if (++looks_ > 64) std::this_thread::yield();
        else __builtin_ia32_pause();
    }

private:
    uint32_t looks_ = 0;
};

class CopyPool;

// A list of copies, made by run() after the work queued on the stream; run returns when the last byte is in place.
// Held by the object whose stream it uses, so that the pool behind it lives as long as one of them does.
class HostCopies {
public:
    void add(void* dst, const void* src, size_t bytes)
    {
        if (bytes) list_.push_back(Part{ static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src), bytes });
    }
    void run(hipStream_t s);
    // as run, but copies that the device makes by itself (to pinned memory) may be left in flight: true if they are, and
    // without copies it waits for nothing
    bool start(hipStream_t s);
    struct Part {
        uint8_t* dst;
        const uint8_t* src;
        size_t bytes;
    };

private:
    std::vector<Part> list_;
    std::shared_ptr<CopyPool> pool_;
    uint64_t asked_ = 0;  // bytes that a pool would have copied so far, and copied
};

}  // namespace vf
