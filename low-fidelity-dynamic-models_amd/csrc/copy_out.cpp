// A copy into pageable memory goes through the runtime's staging buffer and one thread's memcpy, which also
// takes the page faults of memory the caller has just allocated: 10 GB/s for the 600 MB of a 1,000,000-vehicle
// fleet's records, where the link moves 57 GB/s.  Here several threads each take a part of the array
// through two pinned buffers of their own, so that the link, the faults and the copies of different parts
// overlap.
#include "copy_out.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace lfdm {

namespace {

// 16 buffers of 2 MiB: a part takes about 40 us on the link and ten times that to be copied out by one thread.
// 600 MB (GB/s): 8 threads with parts of 1 MiB 30, of 2 MiB 35; 12 or 16 threads 29 (parts of 0.5 MiB 21).
constexpr int kThreads = 8, kBuffers = 2;
constexpr size_t kPart = size_t(2) << 20;
// Below this the threads' start-up costs more than they save.
constexpr size_t kLeast = size_t(4) << 20;
// Pinning the buffers costs 1 to 2 ms, more than a read of less than 30 MB saves, and a handle that is read once and
// closed would pay it each time: they are pinned for a handle once it has read this much.  Made, run 10 steps, read
// once and closed, pinned at once -> so: 7,000 vehicles 4.1 -> 2.5 ms, 10,000 6.0 -> 4.3, 100,003 43.9 -> 44.0.
constexpr size_t kReadBefore = kThreads * kBuffers * kPart;
// A process on one CPU, whose threads only take turns, copies no less than this in parts either: 100,003 vehicles 6.2 ->
// 5.4 ms there, but 30,000 1.35 -> 1.43 and 10,000 0.45 -> 0.53 (on two CPUs 6.2 -> 3.2, 1.31 -> 0.95, 0.45 -> 0.37).
constexpr size_t kLeastOneCpu = kReadBefore;
// A handle's own small buffer takes 26 us to pin and free, where a read saves 8: the first read of 64 vehicles 42 ->
// 25 us, the fifth 16.
constexpr int kPlainReads = 3;

std::mutex g_lock;  // guards the buffers; a copy holds it, a second one at the time goes the plain way
char* g_pinned = nullptr;
size_t g_parts = 0;  // parts it holds, kThreads x kBuffers at most
// The holders have a lock of their own: handles come and go while a copy is under way.
std::mutex g_holders_lock;
int g_holders = 0;

// One thread's share: every kThreads-th part.
hipError_t copy_parts(int device, char* dst, const char* src, size_t n, int first, hipStream_t stream) {
    hipError_t e = hipSetDevice(device);
    hipEvent_t done[kBuffers] = {};
    for (int b = 0; b < kBuffers && e == hipSuccess; ++b) e = hipEventCreateWithFlags(&done[b], hipEventDisableTiming);
    const size_t parts = (n + kPart - 1) / kPart;
    const auto pinned = [](size_t p) { return g_pinned + p % (kThreads * kBuffers) * kPart; };
    const auto size = [&](size_t p) { return std::min(kPart, n - p * kPart); };
    const auto request = [&](size_t p, int b) {
        hipError_t r = hipMemcpyAsync(pinned(p), src + p * kPart, size(p), hipMemcpyDeviceToHost, stream);
        return r == hipSuccess ? hipEventRecord(done[b], stream) : r;
    };
    int b = 0;
    if (e == hipSuccess && (size_t)first < parts) e = request(first, b);
    for (size_t p = first; p < parts && e == hipSuccess; p += kThreads, b = (b + 1) % kBuffers) {
        if (p + kThreads < parts) e = request(p + kThreads, (b + 1) % kBuffers);
        const hipError_t w = hipEventSynchronize(done[b]);
        if (e == hipSuccess) e = w;
        if (e == hipSuccess) std::memcpy(dst + p * kPart, pinned(p), size(p));
    }
    // no request may still be writing the buffers when they go back
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);
    for (hipEvent_t d : done)
        if (d) (void)hipEventDestroy(d);
    return e;
}

// p as n bytes of pinned memory in place of what it was.
bool pin(char*& p, size_t n) {
    if (p) (void)hipHostFree(p);
    if (hipHostMalloc((void**)&p, n, hipHostMallocPortable) != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();  // the plain way is taken instead
    }
    return p != nullptr;
}

// Whether the runtime knows nothing of dst: neither pinned (which the link reaches without staging) nor
// device memory.
bool ordinary(const void* dst) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, dst) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

bool one_cpu() {
    cpu_set_t mine;
    return sched_getaffinity(0, sizeof(mine), &mine) == 0 && CPU_COUNT(&mine) == 1;
}

hipError_t plain(void* dst, const void* src, size_t n, hipStream_t stream) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
}

}  // namespace

Staging::~Staging() {
    if (p_) (void)hipHostFree(p_);
}

char* Staging::buffer(const void* dst, size_t n) {
    if (n > kStagedBytes || !ordinary(dst) || !lock_.try_lock()) return nullptr;
    if (reads_ < kPlainReads) ++reads_;
    else if (n > n_) n_ = pin(p_, n) ? n : 0;
    if (!p_) lock_.unlock();
    return p_;
}

void Staging::done() { lock_.unlock(); }

hipError_t copy_out(void* dst, const void* device_src, size_t n, hipStream_t stream, size_t& before) {
    int device = 0;
    before = std::min(before + n, kReadBefore);
    if (n < (one_cpu() ? kLeastOneCpu : kLeast) || before < kReadBefore || !ordinary(dst) ||
        hipGetDevice(&device) != hipSuccess)
        return plain(dst, device_src, n, stream);
    // The source is complete before a helper is started: hipStreamPerThread names another stream in every
    // thread, on which a helper's copy would not wait for the work ahead on the caller's.  And the buffers
    // are not held, nor do eight threads wait, while that work runs.
    if (const hipError_t e = hipStreamSynchronize(stream); e != hipSuccess) return e;
    std::unique_lock<std::mutex> lock(g_lock, std::try_to_lock);
    if (!lock) return plain(dst, device_src, n, stream);
    const size_t parts = std::min<size_t>((n + kPart - 1) / kPart, kThreads * kBuffers);
    if (parts > g_parts) g_parts = pin(g_pinned, parts * kPart) ? parts : 0;
    if (!g_pinned) return plain(dst, device_src, n, stream);
    hipError_t result[kThreads];
    std::vector<std::thread> helpers;
    int started = 1;  // this thread takes the first share
    try {
        helpers.reserve(kThreads);
        for (; started < kThreads; ++started)
            helpers.emplace_back([&, k = started] {
                result[k] = copy_parts(device, (char*)dst, (const char*)device_src, n, k, stream);
            });
    } catch (...) {  // no more threads: the shares left over are this thread's too
    }
    result[0] = copy_parts(device, (char*)dst, (const char*)device_src, n, 0, stream);
    for (int k = started; k < kThreads; ++k)
        result[k] = copy_parts(device, (char*)dst, (const char*)device_src, n, k, stream);
    for (std::thread& t : helpers) t.join();
    for (hipError_t e : result)
        if (e != hipSuccess) {  // what failed (an event, say) the plain way may not need
            (void)hipGetLastError();
            return plain(dst, device_src, n, stream);
        }
    return hipSuccess;
}

void copy_out_hold() {
    std::lock_guard<std::mutex> lock(g_holders_lock);
    ++g_holders;
}

void copy_out_release() {
    std::lock_guard<std::mutex> holders(g_holders_lock);
    if (--g_holders > 0) return;
    std::lock_guard<std::mutex> lock(g_lock);  // free: a copy is made for a handle
    if (g_pinned) (void)hipHostFree(g_pinned);
    g_pinned = nullptr;
    g_parts = 0;
}

}  // namespace lfdm
