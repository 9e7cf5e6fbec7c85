// hostcopy.h — copies between the caller's (pageable) host memory and the device.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace hgpm {

// One contiguous piece of a transfer.  check (to the device only): 0 = none, 1 = every
// float finite, 2 = every float below 2^30 in magnitude (and not NaN).  scratch: host memory
// that the calling thread has just written and will write again on its next call.
struct HostSeg {
    void* host;
    void* dev;
    size_t bytes;
    int check = 0;
    bool scratch = false;
};

// Move the segments in order through a ring of pinned slots, the memory copies by several
// threads beside the transfers (uploads of a middle size take the runtime's own copy); both
// return after the data has arrived.  The runtime's own
// copy from or to pageable memory pins the caller's pages on each call, on one thread.
// Measured, reading back 128^3 particles (50 MB, fresh memory): 5.5 ms, through the ring
// 1.4-1.7 ms; 32^3 particles (0.8 MB): 0.37 ms, now 0.08 ms.
// Page-locked memory of the caller's is left to the copy engine (57 GB/s; through the ring
// 2 MB come back in 121 us instead of 45, 128 MB in 3.5 ms instead of 2.4).
// bad: the first segment with a value that fails its check, or -1; every segment is
// transferred all the same.
// st is a stream of `device`, which need not be the calling thread's current device.
hipError_t copy_to_host(const HostSeg* seg, int n, int device, hipStream_t st);
hipError_t copy_to_device(const HostSeg* seg, int n, int device, hipStream_t st, int* bad);

// Rings are 16 MB, one per transfer under way; up to two idle ones are kept between
// transfers, while any context lives (add and release one owner each).  Where the host
// cannot pin one the segments take the runtime's own copy.
void host_copy_add_owner();
void host_copy_release_owner();

} // namespace hgpm
