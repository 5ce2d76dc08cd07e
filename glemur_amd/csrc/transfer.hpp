// Copies between a caller's (pageable) arrays and device memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace gm {

// Staging memory is shared by the contexts of the process: taken at the
// first large copy, given back when the last context is destroyed.
void staging_retain();
void staging_release();

// dst (device) <- src (host), ordered on s; src must stay as it is until s has
// been waited for (a copy from pinned memory may still be under way on return)
hipError_t copy_to_device(hipStream_t s, void *dst, const void *src, size_t bytes);
// dst (host) <- src (device) after the work on s; complete on return
hipError_t copy_to_host(hipStream_t s, void *dst, const void *src, size_t bytes);

}  // namespace gm
