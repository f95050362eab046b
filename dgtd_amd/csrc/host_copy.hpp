// State vectors between the device (FP64 or FP32) and host FP64 arrays.
//
// A large vector goes through a ring of pinned blocks: the copy engine moves
// one block while worker threads convert and copy others.  A plain
// hipMemcpy to or from the caller's pageable array is staged by one thread of
// the runtime (about 10 GB/s), an FP32 vector then needed a second whole
// host vector and one more pass by the calling thread, and the first touch of
// a fresh destination, page by page, stays on that thread too.  Measured for
// 41.3 million FP32 unknowns (165 MB on the device, 330 MB on the host):
// download 59 ms -> 6.1 ms, upload 38 -> 5.7 ms (FP64 download 32 -> 11 ms; FP64
// uploads, which convert nothing, stay plain copies).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace dgtd {

// The transfers of one operator or batch, from any threads.  Each borrows a
// ring of pinned blocks; the process keeps at most two idle ones and frees them
// with the last HostCopy.
class HostCopy {
public:
    HostCopy();
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;
    ~HostCopy();

    // h[i] = d[i], after the work queued on s; returns when h is complete.
    template <typename T>
    hipError_t to_host(const T* d, double* h, int64_t n, hipStream_t s);
    // d[i] = h[i] on s; h stays valid until s has drained.
    template <typename T>
    hipError_t to_device(const double* h, T* d, int64_t n, hipStream_t s);
};

}  // namespace dgtd
