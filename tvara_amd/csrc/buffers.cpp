// Device and pinned host buffers, and the plan pool (see buffers.hpp).
#include "buffers.hpp"

#include <algorithm>
#include <array>

namespace tvara_amd {

namespace {
size_t pages(size_t n) { return (n + 4095) / 4096 * 4096; }
}  // namespace

void* DeviceBuffer::ensure(size_t n) {
    if (n <= bytes && ptr) return ptr;
    if (ptr) {
        TVARA_HIP(hipDeviceSynchronize());
        TVARA_HIP(hipFree(ptr));
        ptr = nullptr;
        bytes = 0;
    }
    const size_t want = std::max<size_t>(pages(n), 4096);
    TVARA_HIP(hipMalloc(&ptr, want));
    bytes = want;
    return ptr;
}

DeviceBuffer::~DeviceBuffer() {
    if (ptr) (void)hipFree(ptr);
}

void* PinnedBuffer::acquire(size_t n) {
    if (done) TVARA_HIP(hipEventSynchronize(done));
    if (n > bytes || !ptr) {
        if (ptr) TVARA_HIP(hipHostFree(ptr));
        ptr = nullptr;
        const size_t want = std::max<size_t>(pages(n), 4096);
        TVARA_HIP(hipHostMalloc(&ptr, want, hipHostMallocDefault));
        bytes = want;
    }
    return ptr;
}

void PinnedBuffer::release(hipStream_t s) {
    if (!done) TVARA_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    TVARA_HIP(hipEventRecord(done, s));
}

PinnedBuffer::~PinnedBuffer() {
    if (done) {
        (void)hipEventSynchronize(done);
        (void)hipEventDestroy(done);
    }
    if (ptr) (void)hipHostFree(ptr);
}

PlanPool::Set::~Set() {
    if (idle) (void)hipEventDestroy(idle);
}

std::unique_ptr<PlanPool::Set> PlanPool::take(size_t bytes) {
    int device = 0;
    TVARA_HIP(hipGetDevice(&device));
    std::unique_ptr<Set> out;
    // An event that is not ready leaves that as the runtime's last error, which
    // is cleared; an error that waits there already, or any other answer of a
    // query, is for the caller's next check.
    if (hipPeekAtLastError() == hipSuccess) {
        std::lock_guard<std::mutex> hold(lock_);
        size_t best = sets_.size();
        for (size_t i = 0; i < sets_.size(); ++i) {
            if (sets_[i]->device != device || sets_[i]->region.bytes < bytes ||
                (best < sets_.size() && sets_[i]->region.bytes >= sets_[best]->region.bytes))
                continue;
            const hipError_t e = hipEventQuery(sets_[i]->idle);
            if (e == hipSuccess) best = i;
            if (e == hipErrorNotReady) (void)hipGetLastError();
        }
        if (best < sets_.size()) {
            out = std::move(sets_[best]);
            sets_.erase(sets_.begin() + static_cast<std::ptrdiff_t>(best));
        }
    }
    if (!out) {
        // the event is made here, where the plan's device is the current one: a
        // plan may be closed with another one current
        out = std::make_unique<Set>();
        out->device = device;
        TVARA_HIP(hipEventCreateWithFlags(&out->idle, hipEventDisableTiming));
    }
    return out;
}

void PlanPool::give(std::unique_ptr<Set> s) noexcept {
    int device = -1;
    bool marked = s->region.bytes <= kBytes && s->idle && hipGetDevice(&device) == hipSuccess && device == s->device;
    if (marked) {
        // a record that fails (a stream that the null stream waits for is being
        // captured, say) only means that the set is freed: no later check's error
        const bool clean = hipPeekAtLastError() == hipSuccess;
        marked = hipEventRecord(s->idle, nullptr) == hipSuccess;
        if (!marked && clean) (void)hipGetLastError();
    }
    std::array<std::unique_ptr<Set>, kSets + 1> gone;  // freed outside the lock (hipFree waits for a set's work)
    if (marked) {
        std::lock_guard<std::mutex> hold(lock_);
        if (!closed_) {
            sets_.push_back(std::move(s));
            size_t bytes = 0;
            for (const auto& k : sets_) bytes += k->region.bytes;
            for (size_t i = 0; sets_.size() > kSets || bytes > kBytes; ++i) {
                bytes -= sets_.front()->region.bytes;
                gone[i] = std::move(sets_.front());
                sets_.erase(sets_.begin());
            }
        }
    }
}

void PlanPool::clear() {
    std::array<std::unique_ptr<Set>, kSets> gone;
    std::lock_guard<std::mutex> hold(lock_);
    std::move(sets_.begin(), sets_.end(), gone.begin());
    sets_.clear();
}

void PlanPool::close() {
    {
        std::lock_guard<std::mutex> hold(lock_);
        closed_ = true;
    }
    clear();
}

}  // namespace tvara_amd
