// Download of fields from the device.
//
// What bounds it is the host: the link carries 55 GB/s, while one thread that
// lets the runtime stage a pageable copy into a fresh temporary and then
// converts it writes every page three times and faults it in twice (the four
// fields of a 256^3 float lattice: 96 ms, of which the link needs 5). From 16 MB
// on, copies go into page-locked slots, all in flight, and are converted from there
// into place; the destination is faulted in while the stream still computes, which
// is half of the time (after an idle stream, staging and slots: 16 MB float 4.3 and
// 2.4 ms, 30 MB 7.7 and 4.7, 125 MB 25 and 19, 17 MB double 1.14 and 0.80). From
// 128 MB on 4 threads share the chunks: those four fields then take 12 ms (134 MB
// double 4.8 where staging takes 14). Smaller downloads stay on one thread: with
// threads a pass of 9 ms and 28 MB took 11.4 or 23 ms, run by run, beside a caller's
// own spinning pool; between 28 and 125 MB the line was not measured. Below 16 MB
// the runtime's staging is the faster one (0.6 million float nodes 1.4 ms, slots 1.2
// to 2.0).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace vlbm {
namespace detail {

struct FieldCopy {
    const void* dev;      // n values of 4 or 8 bytes on the device
    void* out;            // on the host: n doubles, or n values as they are on the device
};

// Downloads from 16 MB on take slots of a pool that all lattices and batches of
// the process share: 4 of 2 MB for a device, page-locked by the first download
// that needs them and kept until the process ends. Page-locking and first touching
// 8 MB takes up to 3 ms, as long as the download of 16 to 40 MB itself, so slots of
// a handle's own made the first download of a new lattice up to twice as long.
// Downloads at once from several threads hold different slots; those beyond 4 are
// freed at the end of their download.
class HostCopy {
public:
    // The fields, after everything enqueued on the stream so far; returns when they are in place. As doubles, or
    // raw as they are on the device.
    static hipError_t fetch(int device, hipStream_t stream, const FieldCopy* fields, int count, size_t n,
                            int value_bytes, bool raw = false);

private:
    static hipError_t fetch_small(hipStream_t stream, const FieldCopy* fields, int count, size_t n, int value_bytes, bool raw);
};

// out[k] = in[k] for n values of 4 or 8 bytes.
void widen(double* out, const void* in, size_t n, int value_bytes);

}  // namespace detail
}  // namespace vlbm
