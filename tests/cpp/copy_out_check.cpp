// Record copies to the host (csrc/copy_out.cpp) on a stand-in for the HIP runtime: streams are queues of work
// that runs when a thread waits for it, hipStreamPerThread names another queue in every thread, and device
// memory is host memory.  Built without the HIP library by the Makefile's `copycheck`; run by
// tests/test_copy_out_host.py, one check per argument.
#include "../../low-fidelity-dynamic-models_amd/csrc/copy_out.cpp"

#include <sched.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <map>
#include <string>

namespace {

struct Queue {
    std::mutex lock, running;
    std::deque<std::function<void()>> work;
    void add(std::function<void()> f) {
        std::lock_guard<std::mutex> g(lock);
        work.push_back(std::move(f));
    }
    // Runs the queue in order until done() (null: until it is empty).
    void drain(const std::function<bool()>& done) {
        std::lock_guard<std::mutex> one(running);
        while (!done || !done()) {
            std::function<void()> f;
            {
                std::lock_guard<std::mutex> g(lock);
                if (work.empty()) return;
                f = std::move(work.front());
                work.pop_front();
            }
            f();
        }
    }
};

Queue& queue_of(hipStream_t s) {
    if (s == hipStreamPerThread) {
        static thread_local Queue own;
        return own;
    }
    return *reinterpret_cast<Queue*>(s);
}

struct Event {
    std::atomic<bool> done{true};
    Queue* queue = nullptr;
};

std::mutex g_count_lock;
std::map<void*, size_t> g_allocated;  // pinned blocks alive
int g_pins = 0;                       // pinned blocks ever
std::atomic<int> g_copies{0};         // copies asked of the runtime
std::atomic<int> g_events_left{1 << 30};  // events the runtime can still make

}  // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (g_events_left-- <= 0) return hipErrorOutOfMemory;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Event* ev = reinterpret_cast<Event*>(e);
    ev->queue = &queue_of(s);
    ev->done = false;
    ev->queue->add([ev] { ev->done = true; });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Event* ev = reinterpret_cast<Event*>(e);
    if (ev->queue) ev->queue->drain([ev] { return ev->done.load(); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    queue_of(s).drain(nullptr);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    ++g_copies;
    queue_of(s).add([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    std::lock_guard<std::mutex> g(g_count_lock);
    g_allocated[*p] = n;
    ++g_pins;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> g(g_count_lock);
    if (!g_allocated.erase(p)) std::abort();
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    *a = {};
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
}

namespace {


constexpr size_t kMiB = size_t(1) << 20;

// A copy for a handle that has read nothing before.
hipError_t copy_out(void* dst, const void* src, size_t n, hipStream_t stream) {
    size_t before = 0;
    return lfdm::copy_out(dst, src, n, stream, before);
}

std::vector<char> bytes(size_t n, int seed) {
    std::vector<char> v(n);
    unsigned x = seed * 2654435761u + 1;
    for (char& c : v) c = (char)((x = x * 1664525u + 1013904223u) >> 24);
    return v;
}

// Work ahead of the copy, on the calling thread's hipStreamPerThread: every byte must come from after it.
bool per_thread_stream() {
    const std::vector<char> fresh = bytes(33 * kMiB + 7, 1);
    std::vector<char> device(fresh.size(), 'x'), out(fresh.size());
    queue_of(hipStreamPerThread).add([&] {
        std::this_thread::sleep_for(std::chrono::milliseconds(200));
        device = fresh;
    });
    return copy_out(out.data(), device.data(), out.size(), hipStreamPerThread) == hipSuccess && out == fresh;
}

// A copy that still waits for work ahead of it keeps neither the pinned parts nor the helper threads: one of a
// finished stream meanwhile goes in parts.
bool waiting_copy_keeps_nothing() {
    const std::vector<char> fresh = bytes(40 * kMiB, 2);
    std::vector<char> a(fresh.size()), b(fresh.size());
    Queue busy, idle;
    std::atomic<bool> reached{false}, go{false};
    busy.add([&] {
        reached = true;
        while (!go) std::this_thread::yield();
    });
    bool ok = true;
    std::thread waits([&] {
        ok = copy_out(a.data(), fresh.data(), a.size(), reinterpret_cast<hipStream_t>(&busy)) == hipSuccess;
    });
    while (!reached) std::this_thread::yield();
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    const int before = g_copies;
    const bool second = copy_out(b.data(), fresh.data(), b.size(), reinterpret_cast<hipStream_t>(&idle)) == hipSuccess;
    const int parts = g_copies - before;
    go = true;
    waits.join();
    return ok && second && a == fresh && b == fresh && parts == 20;
}

// Two handles' small read backs under way at once each have pinned memory of their own; a second one of the same
// handle has none meanwhile.  A later, larger one has enough.
bool small_reads_apart() {
    std::vector<char> dst(1000);
    lfdm::Staging a, b;
    for (int i = 0; i < 4; ++i)
        for (lfdm::Staging* s : {&a, &b})
            if (s->buffer(dst.data(), dst.size())) s->done();
    char* const p = a.buffer(dst.data(), dst.size());
    char *q = nullptr, *again = p;
    std::thread([&] {
        q = b.buffer(dst.data(), dst.size());
        again = a.buffer(dst.data(), dst.size());
        if (q) std::memset(q, 2, 1000);
        b.done();
    }).join();
    if (!p || !q || again) return false;
    std::memset(p, 1, 1000);
    a.done();
    if (a.buffer(dst.data(), 10) != p || b.buffer(dst.data(), lfdm::kStagedBytes + 1)) return false;
    a.done();
    char* const large = b.buffer(dst.data(), lfdm::kStagedBytes);
    std::memset(large, 3, lfdm::kStagedBytes);
    b.done();
    return true;
}

// A handle that reads little before it goes pins nothing.
bool read_once_pins_nothing() {
    std::vector<char> small(1000), large(5 * kMiB), device(5 * kMiB, 'd');
    Queue idle;
    lfdm::Staging handle;
    size_t before = 0;
    for (int i = 0; i < 2; ++i) {
        if (handle.buffer(small.data(), small.size())) handle.done();
        if (lfdm::copy_out(large.data(), device.data(), large.size(), reinterpret_cast<hipStream_t>(&idle), before) !=
                hipSuccess ||
            large != device)
            return false;
    }
    return g_pins == 0;
}

// One that goes on reading pins what its reads need, once; a larger read of another handle then pins more.
bool later_reads_pin_once() {
    Queue idle;
    size_t first = 0, second = 0;
    const auto read = [&](size_t n, size_t& before) {
        const std::vector<char> device = bytes(n, (int)n);
        std::vector<char> out(n);
        return lfdm::copy_out(out.data(), device.data(), n, reinterpret_cast<hipStream_t>(&idle), before) == hipSuccess &&
               out == device;
    };
    bool ok = true;
    for (int i = 0; i < 12; ++i) ok = ok && read(5 * kMiB + 1, first);
    ok = ok && g_pins == 1 && g_allocated.begin()->second == 6 * kMiB;
    ok = ok && read(19 * kMiB, second) && g_pins == 1;  // this handle's first: the plain way
    ok = ok && read(19 * kMiB, second) && g_pins == 2 && g_allocated.begin()->second == 20 * kMiB;
    ok = ok && read(70 * kMiB + 3, second) && g_pins == 3 && g_allocated.begin()->second == 32 * kMiB;
    return ok && read(5 * kMiB, first) && g_pins == 3 && g_allocated.size() == 1;
}

// A process on one CPU, where helper threads only take turns, copies 18 MB the plain way and 60 MB in parts.
bool one_cpu() {
    cpu_set_t all, one;
    sched_getaffinity(0, sizeof(all), &all);
    CPU_ZERO(&one);
    for (int c = 0; c < CPU_SETSIZE && CPU_COUNT(&one) == 0; ++c)
        if (CPU_ISSET(c, &all)) CPU_SET(c, &one);
    sched_setaffinity(0, sizeof(one), &one);
    Queue idle;
    bool ok = true;
    for (size_t n : {size_t(18000000), size_t(60000000)}) {
        const std::vector<char> device = bytes(n, 9);
        std::vector<char> out(n);
        const int copies = g_copies;
        size_t before = 100 * kMiB;
        ok = ok && lfdm::copy_out(out.data(), device.data(), n, reinterpret_cast<hipStream_t>(&idle), before) == hipSuccess &&
             out == device && g_copies - copies == (n == 18000000 ? 1 : 29);
    }
    return ok;
}

// Without events for some of the parts the copy is made the plain way, which needs none.
bool no_events() {
    Queue idle;
    const std::vector<char> device = bytes(40 * kMiB, 4);
    for (int left : {0, 5, 15}) {
        g_events_left = left;
        std::vector<char> out(device.size());
        if (copy_out(out.data(), device.data(), out.size(), reinterpret_cast<hipStream_t>(&idle)) != hipSuccess ||
            out != device)
            return false;
    }
    return true;
}

}  // namespace

int main(int argc, char** argv) {
    const std::map<std::string, bool (*)()> checks = {{"per_thread_stream", per_thread_stream},
                                                      {"waiting_copy_keeps_nothing", waiting_copy_keeps_nothing},
                                                      {"small_reads_apart", small_reads_apart},
                                                      {"read_once_pins_nothing", read_once_pins_nothing},
                                                      {"later_reads_pin_once", later_reads_pin_once},
                                                      {"one_cpu", one_cpu},
                                                      {"no_events", no_events}};
    const auto it = checks.find(argc > 1 ? argv[1] : "");
    if (it == checks.end()) return 2;
    lfdm::copy_out_hold();
    bool ok = it->second();
    lfdm::copy_out_release();
    ok = ok && g_allocated.empty();
    std::printf("%s %s\n", it->first.c_str(), ok ? "ok" : "FAILED");
    return ok ? 0 : 1;
}
