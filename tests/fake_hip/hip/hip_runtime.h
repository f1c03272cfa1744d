// A stand-in for the HIP runtime on the CPU, for tests of host code that only
// queues copies and events.  One stream: its work is done in order by one
// thread, which waits at a gate (work queued before: the frame being rendered)
// until fake::open() is called.  Calls can be made to fail.
#pragma once
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
using hipStream_t = int;

namespace fake {

inline std::mutex mu;
inline std::condition_variable cv;
inline std::deque<std::function<void()>> queue;
inline bool is_open = false, quit = false, idle = true;
inline int helpers = 0;                  // threads that set their device
inline int waiting = 0, most_waiting = 0;   // threads in hipEventSynchronize while the gate was closed
inline bool no_pinned = false;           // hipHostMalloc fails
inline int fail_copy = -1, fail_sync = -1;   // the n-th copy / event wait from now fails
inline const void* known = nullptr;      // the caller's pinned memory
inline int copies = 0;
inline int pinned = 0, events = 0;       // allocated and not yet given back

inline void work() {
    std::unique_lock<std::mutex> lk(mu);
    for (;;) {
        cv.wait(lk, [] { return quit || (is_open && !queue.empty()); });
        if (quit) return;
        auto f = std::move(queue.front());
        queue.pop_front();
        idle = false;
        lk.unlock();
        f();
        lk.lock();
        idle = true;
        cv.notify_all();
    }
}
inline void push(std::function<void()> f) {
    std::lock_guard<std::mutex> lk(mu);
    queue.push_back(std::move(f));
    cv.notify_all();
}
inline void open(bool on) {
    std::lock_guard<std::mutex> lk(mu);
    is_open = on;
    cv.notify_all();
}
inline bool counted_down(int& n) {
    std::lock_guard<std::mutex> lk(mu);
    return n >= 0 && n-- == 0;
}

struct Event {
    bool done = true;
};

}  // namespace fake

using hipEvent_t = fake::Event*;

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (fake::no_pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    fake::pinned++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::free(p);
    fake::pinned--;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new fake::Event;
    fake::events++;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    fake::events--;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    {
        std::lock_guard<std::mutex> lk(fake::mu);
        e->done = false;
    }
    fake::push([e] {
        std::lock_guard<std::mutex> lk(fake::mu);
        e->done = true;
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (fake::counted_down(fake::fail_sync)) return hipErrorUnknown;
    std::unique_lock<std::mutex> lk(fake::mu);
    fake::waiting++;
    if (!fake::is_open && fake::waiting > fake::most_waiting) fake::most_waiting = fake::waiting;
    fake::cv.wait(lk, [e] { return e->done; });
    fake::waiting--;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (fake::counted_down(fake::fail_copy)) return hipErrorUnknown;
    fake::copies++;
    fake::push([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
    std::unique_lock<std::mutex> lk(fake::mu);
    fake::cv.wait(lk, [] { return fake::idle && fake::queue.empty(); });
    return hipSuccess;
}
inline hipError_t hipSetDevice(int) {
    std::lock_guard<std::mutex> lk(fake::mu);
    fake::helpers++;
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = p == fake::known ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
