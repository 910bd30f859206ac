// Checks of csrc/host_copy.cpp over the model of the HIP runtime; argv[1] names one.
#include <sys/mman.h>
#include <sys/resource.h>

#include <cstdio>
#include <string>
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

}  // namespace

int main(int, char** argv) {
    const std::string name = argv[1];
    if (name == "other_device") return other_device();
    return fail("unknown check");
}
