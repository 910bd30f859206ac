// Current device of the calling thread, for the length of a call.
#pragma once
#include <hip/hip_runtime.h>

namespace vlbm {
namespace detail {

// Makes a device current and restores the caller's. Events and page-locked
// memory belong to the device that is current when they are made, and an event
// is recorded on streams of its own device only.
struct DeviceScope {
    int prev = -1;
    bool ok = false;
    explicit DeviceScope(int device) {
        if (hipGetDevice(&prev) != hipSuccess) return;
        ok = prev == device || hipSetDevice(device) == hipSuccess;
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;
    ~DeviceScope() {
        if (ok && prev >= 0) (void)hipSetDevice(prev);
    }
};

}  // namespace detail
}  // namespace vlbm
