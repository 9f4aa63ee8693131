// Device to host copies of arrays into the caller's ordinary (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace lfdm {

// Copies n bytes from device memory to dst after the work pending on `stream`, and returns when they are
// there.  dst may be any memory hipMemcpy takes; ordinary host memory is the case this is for.  before: what
// the handle has read so far (0 at its start), counted here.
hipError_t copy_out(void* dst, const void* device_src, size_t n, hipStream_t stream, size_t& before);

// A handle's own pinned memory for its small arrays, which a kernel may write itself.  Not shared: a read back
// that waits for work ahead of it keeps no other handle's from its own.
constexpr size_t kStagedBytes = size_t(1) << 20;
class Staging {
public:
    Staging() = default;
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    ~Staging();
    // A buffer of n bytes for dst, the caller's until done(); null where there is none (n above kStagedBytes, dst
    // not ordinary host memory, another thread's read back of the handle under way, the handle's first reads).
    char* buffer(const void* dst, size_t n);
    void done();

private:
    std::mutex lock_;
    char* p_ = nullptr;
    size_t n_ = 0;
    int reads_ = 0;
};

// Solver handles hold copy_out's buffers: the last one to go frees them.
void copy_out_hold();
void copy_out_release();

}  // namespace lfdm
