#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace hfg {
// Copies bytes from the device to pageable host memory, after the work enqueued on st; returns when the
// copy is complete.
hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t st);
}  // namespace hfg
