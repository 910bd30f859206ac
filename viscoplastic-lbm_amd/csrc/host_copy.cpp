// Field downloads (host_copy.h).
#include "host_copy.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "device_scope.h"

namespace vlbm {
namespace detail {
namespace {

constexpr int kThreads = 4;
constexpr int kSlots = 4;                               // of a download, and kept for a device
constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr size_t kStagedBytes = size_t(16) << 20, kThreadBytes = size_t(128) << 20;

// CPUs this process may run on.
int cpus() {
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof(set), &set) == 0) return std::max(1, CPU_COUNT(&set));
    return std::max(1u, std::thread::hardware_concurrency());
}

// fn(0) on this thread, after fn(1) ... fn(workers - 1) have been started on
// their own; fewer when the system refuses a thread. fn must not need them all.
template <typename F>
void run_workers(int workers, F&& fn) {
    std::thread threads[kThreads];
    int started = 0;
    try {
        for (int w = 1; w < workers && w < kThreads; w++) {
            threads[started] = std::thread([&fn, w] { fn(w); });
            started++;
        }
    } catch (...) {
    }
    fn(0);
    for (int t = 0; t < started; t++) threads[t].join();
}

// Writes to every page of [p, p + bytes) without changing it: another thread
// may be storing the values already. The compare-exchange is the first access of
// the page and writes on x86 whatever it finds; a load before it would fault the
// page in for reading first, a second fault a page (30 MB of float fields into
// fresh 4 KB pages after an idle stream: 15.0 ms with the load, 9.5 without,
// 11.9 through the runtime's own staging).
void fault_in(char* p, size_t bytes) {
    for (size_t k = 0; k < bytes; k += 4096) {
        char zero = 0;
        (void)__atomic_compare_exchange_n(p + k, &zero, (char)0, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED);
    }
}

// One page-locked buffer and the event of the copy into it.
struct Slot {
    void* p = nullptr;
    hipEvent_t event = nullptr;
    bool pinned = false;

    bool make() {
        pinned = hipHostMalloc(&p, kSlotBytes, hipHostMallocDefault) == hipSuccess;
        if (!pinned) {
            // pageable memory carries the same copy, staged by the runtime
            (void)hipGetLastError();
            p = std::malloc(kSlotBytes);
        }
        if (p && hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess) return true;
        (void)hipGetLastError();
        event = nullptr;
        drop();
        return false;
    }
    void drop() {
        if (event) (void)hipEventDestroy(event);
        if (pinned) (void)hipHostFree(p);
        else std::free(p);
        *this = Slot();
    }
};

// Slots of a device that no download holds.
class SlotPool {
public:
    // Up to `want` slots of the current device; fewer when the system has no more.
    int take(int device, int want, Slot* out) {
        int got = 0;
        if (device < kDevices) {
            std::lock_guard<std::mutex> lock(mu_);
            while (got < want && count_[device] > 0) out[got++] = idle_[device][--count_[device]];
        }
        while (got < want && out[got].make()) got++;
        return got;
    }
    // Slots that no copy is under way into.
    void give(int device, Slot* slots, int n) {
        for (int k = 0; k < n; k++) {
            if (slots[k].pinned && device < kDevices) {
                std::lock_guard<std::mutex> lock(mu_);
                if (count_[device] < kSlots) {
                    idle_[device][count_[device]++] = slots[k];
                    continue;
                }
            }
            slots[k].drop();
        }
    }

private:
    static constexpr int kDevices = 64;
    std::mutex mu_;
    Slot idle_[kDevices][kSlots];
    int count_[kDevices] = {};
};

// Never destroyed: at the end of the process the runtime may be gone before it.
SlotPool& pool() {
    static SlotPool* p = new SlotPool;
    return *p;
}

// The slots of one download.
struct HeldSlots {
    const int device;
    Slot slot[kSlots];
    const int n;
    HeldSlots(int device_, int want) : device(device_), n(pool().take(device_, std::min(want, kSlots), slot)) {}
    HeldSlots(const HeldSlots&) = delete;
    HeldSlots& operator=(const HeldSlots&) = delete;
    ~HeldSlots() { pool().give(device, slot, n); }
};

}  // namespace

void widen(double* out, const void* in, size_t n, int value_bytes) {
    if (value_bytes == 8) {
        std::memcpy(out, in, n * 8);
        return;
    }
    const float* f = (const float*)in;
    for (size_t k = 0; k < n; k++) out[k] = f[k];
}

// Field by field through the runtime's own staging.
hipError_t HostCopy::fetch_small(hipStream_t stream, const FieldCopy* fields, int count, size_t n, int value_bytes, bool raw) {
    const bool convert = !raw && value_bytes == 4;
    for (int f = 0; f < count; f++) {
        std::vector<float> tmp(convert ? n : 0);
        hipError_t e = hipMemcpyAsync(convert ? (void*)tmp.data() : fields[f].out, fields[f].dev, n * (size_t)value_bytes,
                                      hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return e;
        if (convert) widen((double*)fields[f].out, tmp.data(), n, 4);
    }
    return hipSuccess;
}

hipError_t HostCopy::fetch(int device, hipStream_t stream, const FieldCopy* fields, int count, size_t n,
                           int value_bytes, bool raw) {
    const size_t vb = (size_t)value_bytes, total = n * (size_t)count * vb;
    if (total < kStagedBytes) return fetch_small(stream, fields, count, n, value_bytes, raw);
    const DeviceScope scope(device);         // the caller's current device may be another one
    if (!scope.ok) return hipErrorInvalidDevice;
    // equal chunks of a field, none larger than a slot
    const size_t per_field = (n * vb + kSlotBytes - 1) / kSlotBytes, chunks = per_field * (size_t)count;
    const size_t per = per_field ? (n + per_field - 1) / per_field : 0;                  // values of a chunk
    if (!chunks) return hipSuccess;
    HeldSlots held(device, (int)std::min<size_t>(chunks, kSlots));
    if (!held.n) return fetch_small(stream, fields, count, n, value_bytes, raw);
    hipError_t e = hipSuccess;
    struct Chunk { const char* dev; char* out; size_t n; };
    const size_t ob = raw ? vb : sizeof(double);
    auto chunk = [&](size_t i) {
        const FieldCopy& f = fields[i / per_field];
        const size_t at = i % per_field * per;
        return Chunk{(const char*)f.dev + at * vb, (char*)f.out + at * ob, std::min(per, n - at)};
    };
    auto enqueue = [&](size_t i, int s) {
        const Chunk c = chunk(i);
        const hipError_t ec = hipMemcpyAsync(held.slot[s].p, c.dev, c.n * vb, hipMemcpyDeviceToHost, stream);
        return ec == hipSuccess ? hipEventRecord(held.slot[s].event, stream) : ec;
    };
    auto finish = [&](size_t i, int s) {
        const hipError_t es = hipEventSynchronize(held.slot[s].event);
        if (es != hipSuccess) return es;
        const Chunk c = chunk(i);
        if (raw) std::memcpy(c.out, held.slot[s].p, c.n * vb);
        else widen((double*)c.out, held.slot[s].p, c.n, value_bytes);
        return hipSuccess;
    };
    if (total < kThreadBytes) {
        // all slots in flight; the destination is faulted in while the stream computes
        const size_t ahead = (size_t)held.n;
        for (size_t i = 0; i < std::min(ahead, chunks) && e == hipSuccess; i++) e = enqueue(i, (int)i);
        for (size_t i = 0; i < chunks && e == hipSuccess; i++) fault_in(chunk(i).out, chunk(i).n * ob);
        for (size_t i = 0; i < chunks && e == hipSuccess; i++) {
            e = finish(i, (int)(i % ahead));
            if (e == hipSuccess && i + ahead < chunks) e = enqueue(i + ahead, (int)(i % ahead));
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);      // no copy into a slot outlives the call
        return e;
    }
    std::atomic<size_t> touch{0}, next{0};
    std::atomic<int> error{(int)hipSuccess};
    std::atomic<bool> ready{false};
    std::mutex m;
    std::condition_variable cv;
    auto worker = [&](int w) {
        hipError_t we = hipSuccess;
        if (w == 0) {
            we = hipStreamSynchronize(stream);
            {
                std::lock_guard<std::mutex> g(m);
                ready = true;
            }
            cv.notify_all();
        } else {
            we = hipSetDevice(device);
            // the pages of the destination, while the stream computes
            for (size_t i; !ready && (i = touch++) < chunks;) {
                const Chunk c = chunk(i);
                fault_in(c.out, c.n * ob);
            }
            std::unique_lock<std::mutex> g(m);
            cv.wait(g, [&] { return ready.load(); });
        }
        for (size_t i; we == hipSuccess && error == (int)hipSuccess && (i = next++) < chunks;) {
            we = enqueue(i, w);
            if (we == hipSuccess) we = finish(i, w);
        }
        if (we != hipSuccess) error = (int)we;
    };
    run_workers(std::min({held.n, kThreads, cpus()}), worker);
    // a copy of a worker that stopped early may still be under way into its slot
    if (error != (int)hipSuccess) (void)hipStreamSynchronize(stream);
    return (hipError_t)error.load();
}

}  // namespace detail
}  // namespace vlbm
