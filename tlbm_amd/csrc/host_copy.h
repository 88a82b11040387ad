// host_copy.h -- copies of device memory into a caller's pageable arrays.
//
// The runtime's own copy into pageable memory goes through one staging buffer
// and one host thread (16 GB/s measured on an MI355X host; a pinned copy runs
// at 57).  A long copy here goes in chunks through a ring of pinned slots:
// while the DMA engine fills some, host threads empty the others into the
// caller's array, widening FP32 values to double on the way and sharing the
// page faults of a fresh array.  us per call, before and after: moments of
// 192^3 nodes in FP32 43000 -> 6200, of 128^3 12300 -> 2300 to 6400 (fresh
// arrays); FP64 populations of 64^3 D3Q19 nodes 3900 -> 2200, of 96^3
// 12700 -> 7500.  Uploads stay with the runtime, which takes pageable memory
// faster (192^3 initial moments 7.0 ms, through a ring 12).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace tlbm {

// `count` values at `dev` (FP32 if the copy widens, else doubles) to the
// doubles at `host`.
struct CopyPart {
    const char *dev;
    double *host;
    size_t count;
};

// Copies n parts in the order of a stream of `device` and returns when the
// host has the values.  The calling thread's device does not matter.
hipError_t copy_to_host(const CopyPart *parts, int n, bool widen, hipStream_t stream, int device);

// Rings are kept while any lattice is alive (at most two, of 8 MiB) and given
// back with the last one.
void host_copy_retain();
void host_copy_release();

}  // namespace tlbm
