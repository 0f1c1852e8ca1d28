// Large device-to-host copies into ordinary memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace gc {

// Copies bytes from device memory to dst and returns when dst holds them;
// what st was given before is finished first.  Small copies are one
// hipMemcpy.
hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t st);
// Gives the pinned memory of copy_to_host back (it takes it again on use).
void copy_release();

}  // namespace gc
