// lbm_readback.hpp -- device memory to pageable host memory.
//
// hipMemcpyAsync into pageable memory goes through the runtime's own staging
// on the calling thread: 10 GB/s for the 201 MB of a 4096^2 macro field (19.2
// ms), and 0.41 ms for a single megabyte, which the link carries into pinned
// memory in 27 us (57 GB/s for large copies).  Fresh host pages are the other
// bound: one thread fills them at 4 GB/s where the kernel has to clear them.
//
// Staging keeps a few pinned slots with the handle.  A small readback
// pipelines its chunks through them on the calling thread; a large one
// starts threads that take chunks through a slot of their own each and end
// before the call returns.  4096^2: 7.1 ms, 2048^2: 5.6 to 2.0 ms.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {

struct HostPiece {
    void* dst;        // host memory, nullptr: skipped
    const void* src;  // device memory
    size_t bytes;
};

class Staging {
public:
    Staging() = default;
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    ~Staging()
    {
        for (hipEvent_t e : events_)
            if (e) (void)hipEventDestroy(e);
        if (host_) (void)hipHostFree(host_);
    }

    // Pinned memory for readbacks of `total` bytes at a time, kept until the
    // object ends; called where the object is made, so that the first readback
    // finds it (12 MiB take about 2 ms to pin).
    hipError_t reserve(size_t total)
    {
        const size_t want = std::min(slots_for(total), (total + kSlot - 1) / kSlot);
        for (size_t k = 0; k < want; ++k)
            if (!events_[k])
                if (hipError_t r = hipEventCreateWithFlags(&events_[k], hipEventDisableTiming)) return r;
        if (want <= slots_) return hipSuccess;
        if (host_) (void)hipHostFree(host_);
        host_ = nullptr;
        slots_ = 0;
        if (hipError_t r = hipHostMalloc((void**)&host_, want * kSlot, hipHostMallocDefault)) {
            host_ = nullptr;
            (void)hipGetLastError();  // readbacks go the runtime's way
            return r;
        }
        slots_ = want;
        return hipSuccess;
    }

    // Copies the pieces, in stream order after what `s` holds, and waits.
    hipError_t to_host(const HostPiece* pieces, int count, hipStream_t s, int dev) noexcept
    {
        try {
            return staged(pieces, count, s, dev);
        } catch (...) {  // no memory for the chunk list
            return plain(pieces, count, s);
        }
    }

private:
    hipError_t staged(const HostPiece* pieces, int count, hipStream_t s, int dev)
    {
        size_t total = 0;
        bool direct = false;
        for (int k = 0; k < count; ++k) {
            if (!pieces[k].dst) continue;
            total += pieces[k].bytes;
            direct = direct || known_to_runtime(pieces[k].dst);
        }
        if (total == 0) return hipStreamSynchronize(s);
        if (direct || reserve(total) != hipSuccess) return plain(pieces, count, s);
        std::vector<Chunk> chunks;
        for (int k = 0; k < count;) {
            // a run of pieces that lie one behind the other on the device
            int end = k + 1;
            size_t run = pieces[k].bytes;
            while (end < count && pieces[k].dst && pieces[end].dst &&
                   (const char*)pieces[k].src + run == (const char*)pieces[end].src)
                run += pieces[end++].bytes;
            for (size_t at = 0; pieces[k].dst && at < run; at += kSlot)
                chunks.push_back({pieces + k, at, std::min(kSlot, run - at)});
            k = end;
        }
        return total < kThreaded ? pipelined(chunks, s) : threaded(chunks, s, dev);
    }

    struct Chunk {
        const HostPiece* first;  // of its run
        size_t at, bytes;        // in the run
    };
    static constexpr size_t kSlots = 12, kSlot = 1u << 20;
    // Below 6 MiB one thread and two slots that take turns (the link fills one
    // faster than the thread empties the other), four threads up to 32 MiB,
    // twelve beyond.  One thread and four, microseconds, a program's arrays
    // reused and kept: 5.0 MB 250 to 1180 and 600 to 750; 6.7 MB 1040 to 1400
    // and 720 to 800; 12.6 MB 1490 to 1880 and 900.
    static constexpr size_t kThreaded = 6u << 20, kMore = 32u << 20;
    static constexpr size_t slots_for(size_t total)
    {
        return total < kThreaded ? 2 : (total < kMore ? 4 : kSlots);
    }

    // Memory the runtime has pinned or owns is written directly.
    static bool known_to_runtime(const void* p)
    {
        hipPointerAttribute_t at;
        if (hipPointerGetAttributes(&at, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return at.type != hipMemoryTypeUnregistered;
    }

    static hipError_t plain(const HostPiece* pieces, int count, hipStream_t s)
    {
        (void)hipGetLastError();
        for (int k = 0; k < count; ++k) {
            if (!pieces[k].dst) continue;
            hipError_t e = hipMemcpyAsync(pieces[k].dst, pieces[k].src, pieces[k].bytes, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) return e;
        }
        return hipStreamSynchronize(s);
    }

    hipError_t issue(const Chunk& c, size_t k, hipStream_t s)
    {
        hipError_t e = hipMemcpyAsync(host_ + k * kSlot, (const char*)c.first->src + c.at, c.bytes,
                                      hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipEventRecord(events_[k], s) : e;
    }

    hipError_t take(const Chunk& c, size_t k)
    {
        hipError_t e = hipEventSynchronize(events_[k]);
        if (e == hipSuccess) unload(c, k);
        return e;
    }

    void unload(const Chunk& c, size_t k)
    {
        const char* from = host_ + k * kSlot;
        size_t at = c.at, left = c.bytes;
        for (const HostPiece* p = c.first; left; at = at > p->bytes ? at - p->bytes : 0, ++p) {
            if (at >= p->bytes) continue;
            const size_t n = std::min(left, p->bytes - at);
            std::memcpy((char*)p->dst + at, from, n);
            from += n;
            left -= n;
        }
    }

    hipError_t pipelined(const std::vector<Chunk>& chunks, hipStream_t s)
    {
        const size_t n = chunks.size();
        hipError_t e = hipSuccess;
        size_t issued = 0, taken = 0;
        while (taken < n && e == hipSuccess) {
            while (e == hipSuccess && issued < n && issued < taken + slots_) {
                e = issue(chunks[issued], issued % slots_, s);
                if (e == hipSuccess) ++issued;
            }
            if (e == hipSuccess) e = take(chunks[taken], taken % slots_);
            ++taken;
        }
        const hipError_t w = hipStreamSynchronize(s);  // no copy into a slot outlives the call
        return e != hipSuccess ? e : w;
    }

    // The other threads sleep until the stream has come to the readback: the
    // runtime's waits spin, and twelve of them through a run of 2000 steps at
    // 4096^2 took 1.7 s of processor time in 0.14 s.
    hipError_t threaded(const std::vector<Chunk>& chunks, hipStream_t s, int dev)
    {
        const size_t n = chunks.size();
        const size_t hw = std::max(1u, std::thread::hardware_concurrency());
        const size_t workers = std::min({slots_, n, hw});
        std::atomic<int> error{(int)hipSuccess};
        std::atomic<size_t> next{1};  // chunk 0 is the calling thread's
        std::mutex gate;
        std::condition_variable opened;
        bool open = false;
        auto rest = [&](size_t w, hipError_t e) {
            for (size_t k; e == hipSuccess && error.load() == (int)hipSuccess && (k = next.fetch_add(1)) < n;) {
                e = issue(chunks[k], w, s);
                if (e == hipSuccess) e = take(chunks[k], w);
            }
            if (e != hipSuccess) error.store((int)e);
        };
        auto work = [&](size_t w) {
            {
                std::unique_lock<std::mutex> lock(gate);
                opened.wait(lock, [&] { return open; });
            }
            rest(w, hipSetDevice(dev));
        };
        std::vector<std::thread> threads;
        hipError_t e = issue(chunks[0], 0, s);
        try {
            threads.reserve(workers);
            for (size_t w = 1; w < workers; ++w) threads.emplace_back(work, w);
        } catch (...) {  // no thread to be had: the ones that started, and this one, do the work
        }
        if (e == hipSuccess) e = hipEventSynchronize(events_[0]);
        if (e != hipSuccess) error.store((int)e);
        {
            std::lock_guard<std::mutex> lock(gate);
            open = true;
        }
        opened.notify_all();
        if (e == hipSuccess) unload(chunks[0], 0);
        rest(0, e);
        for (std::thread& t : threads) t.join();
        const hipError_t w = hipStreamSynchronize(s);
        return error.load() != (int)hipSuccess ? (hipError_t)error.load() : w;
    }

    char* host_ = nullptr;
    size_t slots_ = 0;
    hipEvent_t events_[kSlots] = {};
};

}  // namespace lbm
