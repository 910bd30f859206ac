// A model of the few HIP runtime calls that the library's host-only code makes,
// for tests on the CPU: two devices, streams that run nothing before somebody
// waits for them, and the rule that an event is recorded on a stream of its own
// device only.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101, hipErrorInvalidHandle = 400, hipErrorNotReady = 600 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace stub {
constexpr int kDevices = 2;
inline thread_local int device = 0;
inline std::atomic<int> host_allocs{0}, host_live{0};      // page-locked blocks: ever, and now
inline std::atomic<int> events_live{0};
inline std::atomic<bool> refuse_host_malloc{false}, refuse_events{false};

struct Event {
    int device;
    bool recorded = false, done = true;
};
struct Op {
    void* dst;
    const void* src;
    size_t bytes;
    Event* event;       // a record, if not null
};
struct Stream {
    int device;
    std::mutex mu;
    std::deque<Op> ops;
    void drain(const Event* until) {
        std::lock_guard<std::mutex> g(mu);
        while (!ops.empty() && !(until && until->done)) {
            const Op op = ops.front();
            ops.pop_front();
            if (op.event) op.event->done = true;
            else std::memcpy(op.dst, op.src, op.bytes);
        }
    }
};
inline Stream* stream_of_event(const Event* e, Stream* s = nullptr) {
    static std::mutex mu;
    static std::deque<std::pair<const Event*, Stream*>> at;
    std::lock_guard<std::mutex> g(mu);
    for (auto& p : at)
        if (p.first == e) {
            if (s) p.second = s;
            return p.second;
        }
    if (s) at.emplace_back(e, s);
    return s;
}
}  // namespace stub

using hipStream_t = stub::Stream*;
using hipEvent_t = stub::Event*;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetDevice(int* d) { *d = stub::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= stub::kDevices) return hipErrorInvalidDevice;
    stub::device = d;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (stub::refuse_host_malloc) return hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    stub::host_allocs++;
    stub::host_live++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::free(p);
    stub::host_live--;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (stub::refuse_events) return hipErrorOutOfMemory;
    *e = new stub::Event{stub::device};
    stub::events_live++;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    (void)e;                    // kept: stream_of_event goes by its address
    stub::events_live--;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) {
    std::lock_guard<std::mutex> g(s->mu);
    s->ops.push_back({dst, src, bytes, nullptr});
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->device != s->device) return hipErrorInvalidHandle;
    stub::stream_of_event(e, s);
    std::lock_guard<std::mutex> g(s->mu);
    e->recorded = true;
    e->done = false;
    s->ops.push_back({nullptr, nullptr, 0, e});
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->recorded) stub::stream_of_event(e)->drain(e);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->drain(nullptr);
    return hipSuccess;
}
