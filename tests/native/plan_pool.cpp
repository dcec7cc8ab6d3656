// The pool of closed plans' buffers (buffers.cpp) on a stand-in for the HIP
// runtime: two devices, events that end when the test says so, and the
// runtime's habit of keeping the last error for a later hipGetLastError().
#include "buffers.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>

namespace {
int device = 0;
hipError_t last = hipSuccess, record_result = hipSuccess;
std::map<void*, std::pair<int, size_t>> memory;  // device, bytes
struct Event {
    int device;
    bool recorded = false, ended = false;
};
std::set<Event*> events;

hipError_t result(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
hipError_t query_result = hipSuccess;
size_t held(int d) {
    size_t n = 0;
    for (const auto& m : memory)
        if (m.second.first == d) n += m.second.second;
    return n;
}
void end_all() {
    for (Event* e : events) e->ended = true;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return memory[*p = std::malloc(16)] = {device, n}, hipSuccess; }
hipError_t hipFree(void* p) {
    if (!memory.erase(p)) return result(hipErrorInvalidValue);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipDeviceSynchronize() { return end_all(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    auto* made = new Event{device};
    events.insert(made);
    return *e = reinterpret_cast<hipEvent_t>(made), hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    auto* ev = reinterpret_cast<Event*>(e);
    if (record_result != hipSuccess) return result(record_result);
    if (ev->device != device) return result(hipErrorInvalidHandle);
    ev->recorded = true;
    ev->ended = false;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    auto* ev = reinterpret_cast<Event*>(e);
    if (query_result != hipSuccess) return result(query_result);
    return result(ev->recorded && !ev->ended ? hipErrorNotReady : hipSuccess);
}
hipError_t hipEventSynchronize(hipEvent_t e) { return reinterpret_cast<Event*>(e)->ended = true, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) {
    auto* ev = reinterpret_cast<Event*>(e);
    events.erase(ev);
    delete ev;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipPeekAtLastError() { return last; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
}

using tvara_amd::PlanPool;

namespace {
int failures = 0;
void check(bool ok, const char* what) {
    if (!ok) std::printf("failed: %s\n", what);
    failures += !ok;
}

std::unique_ptr<PlanPool::Set> made(PlanPool& pool, size_t bytes) {
    auto s = pool.take(bytes);
    s->region.ensure(bytes);
    return s;
}

void reuse() {
    PlanPool pool;
    auto s = made(pool, 10000);
    PlanPool::Set* first = s.get();
    pool.give(std::move(s));
    check(made(pool, 10000).get() != first, "a set whose work runs is not handed out");
    end_all();
    s = pool.take(20000);
    check(s.get() != first, "a set that is too small is not handed out");
    s = pool.take(8000);
    check(s.get() == first, "a set whose work has ended is handed out");
    s.reset();
    pool.close();
    check(memory.empty() && events.empty(), "a closed pool holds nothing");
    pool.give(made(pool, 10000));
    check(memory.empty() && events.empty(), "a closed pool keeps nothing");
}

// a plan of device 0 closed while device 1 is current: its event would say
// nothing about its own device's work
void devices() {
    PlanPool pool;
    auto s = made(pool, 10000);
    device = 1;
    pool.give(std::move(s));
    check(memory.empty() && events.empty(), "a set closed under another device is freed");
    device = 0;
    pool.give(made(pool, 10000));
    end_all();
    device = 1;
    s = made(pool, 10000);
    check(memory[s->region.ptr].first == 1, "a set goes to plans of its own device");
    device = 0;
    s.reset();
    check(held(0) > 0 && held(1) == 0, "the other device's set stays");
    pool.close();
    last = hipSuccess;
}

// what the pool does is not seen in the last error, and what others left there
// is not lost
void errors() {
    PlanPool pool;
    pool.give(made(pool, 10000));
    made(pool, 10000);
    check(last == hipSuccess, "an event that is not ready is no error");
    end_all();
    last = hipErrorLaunchFailure;
    made(pool, 10000);
    check(last == hipErrorLaunchFailure, "an earlier error stays for its check");
    last = hipSuccess;
    query_result = hipErrorLaunchFailure;
    made(pool, 10000);
    check(last == hipErrorLaunchFailure, "a query's own error stays for the next check");
    query_result = last = hipSuccess;
    auto s = made(pool, 10000);
    record_result = hipErrorStreamCaptureImplicit;
    const size_t before = memory.size();
    pool.give(std::move(s));
    check(memory.size() == before - 1 && last == hipSuccess, "a record that fails frees the set and is no error");
    s = made(pool, 20000);
    last = hipErrorLaunchFailure;
    pool.give(std::move(s));
    check(last != hipSuccess, "an earlier error stays beside it");
    record_result = last = hipSuccess;
    pool.close();
}

// at most four sets and 64 MiB stay, the latest ones; one above that does not
void bounds() {
    PlanPool pool;
    std::unique_ptr<PlanPool::Set> s[6];
    for (auto& x : s) x = made(pool, 10000);
    for (auto& x : s) pool.give(std::move(x));
    check(memory.size() == 4, "four sets stay");
    pool.clear();
    check(memory.empty() && events.empty(), "a cleared pool holds nothing");
    constexpr size_t MiB = size_t(1) << 20;
    for (int i = 0; i < 4; ++i) s[i] = made(pool, 20 * MiB);
    for (int i = 0; i < 4; ++i) pool.give(std::move(s[i]));
    check(held(0) == 60 * MiB, "64 MiB stay at most");
    pool.give(made(pool, 64 * MiB));
    check(held(0) == 64 * MiB, "the latest stays");
    pool.give(made(pool, 65 * MiB));
    check(held(0) == 64 * MiB, "a set above the bound does not come in");
    pool.close();
    check(memory.empty() && events.empty(), "a closed pool holds nothing");
}
}  // namespace

int main() {
    reuse();
    devices();
    errors();
    bounds();
    std::printf("%s\n", failures ? "failed" : "passed");
    return failures != 0;
}
