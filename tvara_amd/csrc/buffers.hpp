// Device and pinned host buffers, and the pool of them that closed plans leave
// (HIP's host API only: tests/native runs it on a stand-in for the runtime).
#pragma once
#include <cstddef>
#include <memory>
#include <mutex>
#include <vector>

#include "hip_check.hpp"

namespace tvara_amd {

// Grow-only device buffer.
struct DeviceBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    void* ensure(size_t n);
    ~DeviceBuffer();
};

// Grow-only pinned host buffer whose reuse waits for the last copy out of it.
struct PinnedBuffer {
    void* ptr = nullptr;
    size_t bytes = 0;
    hipEvent_t done = nullptr;
    void* acquire(size_t n);
    void release(hipStream_t s);
    ~PinnedBuffer();
};

// Buffers of closed decode plans, kept by a cache for its next plans: a
// serving loop makes a plan per step, and allocating and freeing its device
// region and pinned memory, which waits for the device, cost it a quarter of the
// step (MI355X, 32 sequences, 16 layers: 518 -> 379 us with the append).  A set
// is handed out only after the event recorded behind its last plan's work, so
// neither a launch nor a late error flag of the old plan can meet the new one.
// Only plans whose every launch went to the null stream come here: it outlives
// any plan and is never captured; only on the device that they were allocated
// on.  At most kSets sets of at most kBytes together; the oldest are freed.  The
// cache frees the sets when it goes (plans may outlive it), and when a plan finds
// no device memory.
class PlanPool {
public:
    struct Set {
        DeviceBuffer region;
        PinnedBuffer staging, flag;
        int device = -1;  // that region is allocated on and idle belongs to
        hipEvent_t idle = nullptr;
        ~Set();
    };
    // a set whose region holds `bytes` and whose work has ended, or a new one
    std::unique_ptr<Set> take(size_t bytes);
    void give(std::unique_ptr<Set> s) noexcept;
    void clear();  // frees the sets that are here
    void close();  // and keeps none from now on
    PlanPool() { sets_.reserve(kSets + 1); }  // give() allocates nothing: it runs in destructors

private:
    static constexpr size_t kSets = 4, kBytes = size_t(64) << 20;
    std::mutex lock_;
    std::vector<std::unique_ptr<Set>> sets_;  // oldest first
    bool closed_ = false;
};

}  // namespace tvara_amd
