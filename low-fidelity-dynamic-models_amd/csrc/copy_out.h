// Device to host copies of arrays into the caller's ordinary (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace lfdm {

// Copies n bytes from device memory to dst after the work pending on `stream`, and returns when they are
// there.  dst may be any memory hipMemcpy takes; ordinary host memory is the case this is for.
hipError_t copy_out(void* dst, const void* device_src, size_t n, hipStream_t stream);

// Small arrays for dst: a pinned buffer of n bytes that a kernel may write itself, the caller's until
// copy_out_end; null where there is none (n above kStagedBytes, dst not ordinary host memory, a copy under
// way in another thread).
constexpr size_t kStagedBytes = size_t(1) << 20;
char* copy_out_begin(const void* dst, size_t n);
void copy_out_end();

// Solver handles hold the buffers: the last one to go frees them.
void copy_out_hold();
void copy_out_release();

}  // namespace lfdm
