// The few runtime calls lbm_readback.hpp makes, on the CPU: one stream is one
// thread that runs its commands in order and can be held back, pinned memory
// is counted, and calls can be made to fail.
#pragma once

#include <stddef.h>

#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct hipPointerAttribute_t {
    hipMemoryType type;
};

namespace fake {
struct Event {
    std::mutex mu;
    std::condition_variable cv;
    size_t recorded = 0, reached = 0;
};
struct Stream {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> queue;
    size_t pending = 0;
    bool held = false, ends = false;
    std::thread runner{[this] {
        for (;;) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> l(mu);
                cv.wait(l, [this] { return ends || (!held && !queue.empty()); });
                if (queue.empty() || held) return;
                f = std::move(queue.front());
                queue.pop_front();
            }
            f();
            std::lock_guard<std::mutex> l(mu);
            --pending;
            cv.notify_all();
        }
    }};
    ~Stream()
    {
        {
            std::lock_guard<std::mutex> l(mu);
            ends = true;
            held = false;
        }
        cv.notify_all();
        runner.join();
    }
    void push(std::function<void()> f)
    {
        std::lock_guard<std::mutex> l(mu);
        queue.push_back(std::move(f));
        ++pending;
        cv.notify_all();
    }
    void hold(bool on)
    {
        std::lock_guard<std::mutex> l(mu);
        held = on;
        cv.notify_all();
    }
    void drain()
    {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [this] { return pending == 0; });
    }
};
inline std::atomic<size_t> pinned{0}, pinned_most{0}, events{0};
inline std::atomic<int> waiting{0};      // threads inside a wait of the runtime
inline std::atomic<int> waits{0}, records{0};  // calls so far
inline std::atomic<int> fail_pin{0};     // this many pinned allocations fail
inline std::atomic<int> fail_event{0};
inline std::atomic<int> copies_left{-1};  // copies until one fails, -1: none does
struct Wait {
    Wait()
    {
        ++waiting;
        ++waits;
    }
    ~Wait() { --waiting; }
};
}  // namespace fake

using hipStream_t = fake::Stream*;
using hipEvent_t = fake::Event*;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (fake::fail_pin > 0 && fake::fail_pin-- > 0) return hipErrorOutOfMemory;
    size_t* const a = (size_t*)std::malloc(n + 16);
    a[0] = n;
    *p = (char*)a + 16;
    const size_t now = fake::pinned += n;
    for (size_t m = fake::pinned_most; now > m && !fake::pinned_most.compare_exchange_weak(m, now);) {}
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    size_t* const a = (size_t*)((char*)p - 16);
    fake::pinned -= a[0];
    std::free(a);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*)
{
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    if (fake::fail_event > 0 && fake::fail_event-- > 0) return hipErrorOutOfMemory;
    *e = new fake::Event();
    ++fake::events;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    --fake::events;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    size_t at;
    ++fake::records;
    {
        std::lock_guard<std::mutex> l(e->mu);
        at = ++e->recorded;
    }
    s->push([e, at] {
        std::lock_guard<std::mutex> l(e->mu);
        e->reached = at;
        e->cv.notify_all();
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    fake::Wait w;
    std::unique_lock<std::mutex> l(e->mu);
    const size_t at = e->recorded;
    e->cv.wait(l, [e, at] { return e->reached >= at; });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    fake::Wait w;
    s->drain();
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
    if (fake::copies_left >= 0 && fake::copies_left-- <= 0) return hipErrorUnknown;
    st->push([d, s, n] { std::memcpy(d, s, n); });
    return hipSuccess;
}
