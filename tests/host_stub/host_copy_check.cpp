// Checks of csrc/host_copy.cpp over the model of the HIP runtime; argv[1] names one.
#include <sys/mman.h>
#include <sys/resource.h>

#include <atomic>
#include <cstdio>
#include <string>
#include <thread>
#include <vector>

#include "host_copy.h"

using namespace vlbm::detail;

namespace {

// Four float fields of n nodes in "device" memory and their download.
struct Fields {
    size_t n;
    std::vector<float> dev;
    std::vector<double> out;
    std::vector<FieldCopy> list;
    explicit Fields(size_t n_) : n(n_), dev(4 * n_), out(4 * n_) {
        for (size_t k = 0; k < dev.size(); k++) dev[k] = (float)(k % 9973) + 0.25f;
        for (int f = 0; f < 4; f++) list.push_back({dev.data() + f * n, out.data() + f * n});
    }
    bool right() const {
        for (size_t k = 0; k < dev.size(); k++)
            if (out[k] != (double)dev[k]) return false;
        return true;
    }
};

int fail(const char* what) {
    std::printf("%s\n", what);
    return 1;
}

constexpr size_t kOneThread = 1300003, kThreads = 9000001;      // nodes: 20.8 MB and 144 MB in all, no whole chunks

// A caller whose current device is not the one of the stream.
int other_device() {
    for (size_t n : {kOneThread, kThreads}) {
        stub::Stream s{1};
        Fields a(n), b(n);
        HostCopy owner;
        if (hipSetDevice(0) != hipSuccess) return fail("set-up");
        if (owner.fetch(1, &s, a.list.data(), 4, n, 4) != hipSuccess) return fail("download from another device refused");
        if (stub::device != 0) return fail("the caller's device changed");
        if (!a.right()) return fail("wrong values");
        (void)hipSetDevice(1);
        if (owner.fetch(1, &s, b.list.data(), 4, n, 4) != hipSuccess) return fail("later download refused");
        if (!b.right()) return fail("wrong values later");
    }
    return 0;
}

// A download into fresh memory takes one page fault a page: the first access
// of each page is a write.
int page_faults() {
    const size_t n = kOneThread, bytes = 4 * n * sizeof(double);
    char* out = (char*)mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (out == MAP_FAILED) return fail("set-up");
    (void)madvise(out, bytes, MADV_NOHUGEPAGE);
    stub::Stream s{0};
    Fields a(n);
    HostCopy owner;
    if (owner.fetch(0, &s, a.list.data(), 4, n, 4) != hipSuccess) return fail("download");      // touches the slots
    for (int f = 0; f < 4; f++) a.list[f].out = out + f * n * sizeof(double);
    struct rusage before, after;
    getrusage(RUSAGE_SELF, &before);
    if (owner.fetch(0, &s, a.list.data(), 4, n, 4) != hipSuccess) return fail("download");
    getrusage(RUSAGE_SELF, &after);
    const double faults = (double)(after.ru_minflt - before.ru_minflt), pages = bytes / 4096.0;
    std::printf("%.0f faults, %.0f pages\n", faults, pages);
    if (std::memcmp(out, a.out.data(), bytes) != 0) return fail("wrong values");
    return faults <= 1.1 * pages ? 0 : fail("more than one fault a page");
}

// Lattices opened one after the other, as a parameter study does: only the
// first download in the process pays for page-locked memory. Downloads at once
// each have slots of their own; what is kept afterwards is bounded, per device.
int new_owners() {
    for (int k = 0; k < 5; k++) {
        stub::Stream s{k & 1};
        Fields a(k < 3 ? kOneThread : kThreads);
        HostCopy owner;
        if (owner.fetch(k & 1, &s, a.list.data(), 4, a.n, 4) != hipSuccess) return fail("download");
        if (!a.right()) return fail("wrong values");
    }
    std::printf("%d page-locked blocks for two devices\n", stub::host_allocs.load());
    if (stub::host_allocs > 8) return fail("new lattices page-lock memory of their own");
    std::atomic<int> wrong{0};
    std::vector<std::thread> threads;
    for (int k = 0; k < 6; k++)
        threads.emplace_back([&wrong, k] {
            for (int r = 0; r < 3; r++) {
                stub::Stream s{k & 1};
                Fields a(k < 5 ? kOneThread + k : kThreads);
                HostCopy owner;
                if (owner.fetch(k & 1, &s, a.list.data(), 4, a.n, 4) != hipSuccess || !a.right()) wrong++;
            }
        });
    for (auto& t : threads) t.join();
    if (wrong) return fail("wrong values from downloads at once");
    std::printf("%d blocks and %d events kept\n", stub::host_live.load(), stub::events_live.load());
    return stub::host_live <= 8 && stub::events_live <= 8 ? 0 : fail("more kept than 4 slots a device");
}

// Neither page-locked memory nor events to be had: the runtime's staging serves.
int refused() {
    for (int k = 0; k < 3; k++) {
        stub::refuse_host_malloc = k != 1;
        stub::refuse_events = k > 0;
        stub::Stream s{0};
        Fields a(kOneThread);
        HostCopy owner;
        if (owner.fetch(0, &s, a.list.data(), 4, a.n, 4) != hipSuccess) return fail("download refused");
        if (!a.right()) return fail("wrong values");
    }
    return stub::host_live == 0 && stub::events_live == 0 ? 0 : fail("slots that are not page-locked were kept");
}

}  // namespace

int main(int, char** argv) {
    const std::string name = argv[1];
    if (name == "other_device") return other_device();
    if (name == "page_faults") return page_faults();
    if (name == "new_owners") return new_owners();
    if (name == "refused") return refused();
    return fail("unknown check");
}
