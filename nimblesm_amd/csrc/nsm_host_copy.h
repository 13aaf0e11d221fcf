// nsm_host_copy.h -- copies of device memory into a caller's pageable host
// memory (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace nsm {

// `count` doubles at src (device memory of `device`, the stream's device) to
// the caller's dst, after the work already on `stream`; returns when they
// are there.
hipError_t device_to_host(int device, hipStream_t stream, double* dst, const double* src, size_t count);

// The pinned staging memory these copies keep is released with the last
// holder (one per model).
void host_copy_hold();
void host_copy_release();

}  // namespace nsm
