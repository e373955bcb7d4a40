// host_xfer.h -- host fp64 arrays to and from device buffers (host_xfer.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace gonn {

// One array: `rows` rows of d doubles on the host; on the device either the
// same doubles (dp = 0) or fp32 rows of dp >= d floats, zero-padded, rounded
// to nearest even (as a device conversion rounds).
struct HostCopy {
    double* host;  // read by an upload, written by a download
    void* dev;
    size_t rows;
    int d, dp;
};

// Both run on the calling thread's device, queue their copies on s and use
// the host arrays only until they return. An upload's device data is complete
// for work queued on s afterwards; a download returns with the host arrays
// filled, after everything queued on s before it.
hipError_t host_upload(const HostCopy* c, int n, hipStream_t s);
hipError_t host_download(const HostCopy* c, int n, hipStream_t s);

}  // namespace gonn
