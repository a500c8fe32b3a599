// lbm_readback.hpp -- device memory to pageable host memory.
//
// hipMemcpyAsync into pageable memory goes through the runtime's own staging
// on the calling thread: 10 GB/s for the 201 MB of a 4096^2 macro field (19.2
// ms), and 82 us for a single megabyte into pages that are there, which the
// link carries into pinned memory in 27 us (57 GB/s for large copies).  Fresh
// host pages are the other bound: one thread fills them at 4 GB/s where the
// kernel has to clear them (300 us for that megabyte).
//
// Staging copies through pinned slots, which the objects on a device share.  A
// small readback pipelines its chunks through them on the calling thread; a
// large one starts threads that take chunks through a slot of their own each
// and end before the call returns.  4096^2: 6.9 ms, 2048^2: 4.6 to 1.9 ms.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

namespace lbm {

struct HostPiece {
    void* dst;        // host memory, nullptr: skipped
    const void* src;  // device memory
    size_t bytes;
};

// The pinned slots of one device: at most kSlots of 1 MiB, made when a
// readback first asks for them, lent for the length of one call, and freed
// with the last object that read back through them.  Pinning is what costs
// (0.2 ms a slot, once), so objects do not keep their own: a program with a
// thousand lattices pins as much as one with a single one.
class SlotPool {
public:
    static constexpr size_t kSlots = 12, kSlot = 1u << 20;
    struct Slot {
        char* host = nullptr;
        hipEvent_t event = nullptr;
    };

    // nullptr: a device number beyond the table, whose readbacks go the
    // runtime's way
    static SlotPool* of(int dev)
    {
        static SlotPool pools[64];
        return dev >= 0 && dev < 64 ? &pools[dev] : nullptr;
    }

    void attach()
    {
        std::lock_guard<std::mutex> lock(mu_);
        ++users_;
    }
    void detach()
    {
        std::lock_guard<std::mutex> lock(mu_);
        if (--users_) return;
        for (; made_; --made_) (void)hipEventDestroy(slots_[made_ - 1].event);
        for (; blocks_; --blocks_) (void)hipHostFree(block_[blocks_ - 1]);
    }

    // Lends up to `want` slots; fewer, or none, where other threads hold them
    // or memory cannot be pinned.
    size_t lend(Slot** out, size_t want)
    {
        std::lock_guard<std::mutex> lock(mu_);
        size_t n = 0, idle = 0;
        for (size_t k = 0; k < made_; ++k) idle += !lent_[k];
        if (idle < want) grow(std::min(want - idle, kSlots - made_));
        for (size_t k = 0; k < made_ && n < want; ++k) {
            if (lent_[k]) continue;
            lent_[k] = true;
            out[n++] = &slots_[k];
        }
        return n;
    }
    void take_back(Slot* const* in, size_t n)
    {
        std::lock_guard<std::mutex> lock(mu_);
        for (size_t k = 0; k < n; ++k) lent_[in[k] - slots_] = false;
    }

private:
    // More slots, side by side in one allocation (single ones of 1 MiB take 3 %
    // longer to fill); none if there is no memory to pin.
    void grow(size_t count)
    {
        char* host = nullptr;
        if (count == 0) return;
        if (hipHostMalloc((void**)&host, count * kSlot, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();  // the readback goes the runtime's way
            return;
        }
        const size_t before = made_;
        for (; count; --count, ++made_, host += kSlot) {
            Slot& s = slots_[made_];
            if (hipEventCreateWithFlags(&s.event, hipEventDisableTiming) != hipSuccess) break;
            s.host = host;
        }
        if (count) (void)hipGetLastError();
        if (made_ > before) block_[blocks_++] = slots_[before].host;
        else (void)hipHostFree(host);
    }

    std::mutex mu_;
    size_t users_ = 0, made_ = 0, blocks_ = 0;
    Slot slots_[kSlots];
    bool lent_[kSlots] = {};
    char* block_[kSlots] = {};
};
static_assert(std::is_trivially_destructible_v<SlotPool>, "usable while a process ends");

class Staging {
public:
    Staging() = default;
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    ~Staging()
    {
        if (pool_) pool_->detach();
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
        if (direct) return plain(pieces, count, s);
        if (!pool_ && (pool_ = SlotPool::of(dev))) pool_->attach();
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
        const Loan slots(pool_, std::min(slots_for(total), chunks.size()));
        if (slots.count == 0) return plain(pieces, count, s);
        return total < kThreaded ? pipelined(chunks, slots, s) : threaded(chunks, slots, s, dev);
    }

    struct Loan {  // slots of the pool for one call
        SlotPool* const pool;
        SlotPool::Slot* slot[SlotPool::kSlots];
        const size_t count;
        Loan(SlotPool* p, size_t want) : pool(p), slot{}, count(p ? p->lend(slot, want) : 0) {}
        Loan(const Loan&) = delete;
        Loan& operator=(const Loan&) = delete;
        ~Loan()
        {
            if (count) pool->take_back(slot, count);
        }
    };

    struct Chunk {
        const HostPiece* first;  // of its run
        size_t at, bytes;        // in the run
    };
    static constexpr size_t kSlot = SlotPool::kSlot;
    // Below 4 MiB one thread and two slots that take turns (the link fills one
    // faster than the thread empties the other), four threads up to 32 MiB,
    // twelve beyond.  Microseconds through the runtime, with one thread and
    // with four, into pages that are there / that the kernel has to clear:
    //   1.80 MB  115 / 480   95 / 450  114 / 300   5.88 MB 347 / 1570  285 / 1480  268 / 1060
    //   3.15 MB  205 / 880  160 / 825  171 / 628   7.08 MB 450 / 1950   -          320 / 1250
    //   4.32 MB  285 / 1260 224 / 1106 235 / 775  12.58 MB 770 / 3430   -          500 / 2120
    // A page's state is not known here: the line lies where four threads cost
    // nothing into pages that are there (3.15 MB: 7 %; from 4.3 MB on within
    // the scatter), because they save a quarter and more into the others.
    static constexpr size_t kThreaded = 4u << 20, kMore = 32u << 20;
    static constexpr size_t slots_for(size_t total)
    {
        return total < kThreaded ? 2 : (total < kMore ? 4 : SlotPool::kSlots);
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

    static hipError_t copy(const Chunk& c, const SlotPool::Slot& slot, hipStream_t s)
    {
        return hipMemcpyAsync(slot.host, (const char*)c.first->src + c.at, c.bytes, hipMemcpyDeviceToHost, s);
    }

    static hipError_t issue(const Chunk& c, const SlotPool::Slot& slot, hipStream_t s)
    {
        hipError_t e = copy(c, slot, s);
        return e == hipSuccess ? hipEventRecord(slot.event, s) : e;
    }

    static hipError_t take(const Chunk& c, const SlotPool::Slot& slot)
    {
        hipError_t e = hipEventSynchronize(slot.event);
        if (e == hipSuccess) unload(c, slot);
        return e;
    }

    static void unload(const Chunk& c, const SlotPool::Slot& slot)
    {
        const char* from = slot.host;
        size_t at = c.at, left = c.bytes;
        for (const HostPiece* p = c.first; left; at = at > p->bytes ? at - p->bytes : 0, ++p) {
            if (at >= p->bytes) continue;
            const size_t n = std::min(left, p->bytes - at);
            std::memcpy((char*)p->dst + at, from, n);
            from += n;
            left -= n;
        }
    }

    // The last chunk needs no event: the wait for the stream is its own.  A
    // frame's texels of up to 1 MiB are a single chunk, and the event's record
    // and wait cost 7 of its 34 to 76 us.
    static hipError_t pipelined(const std::vector<Chunk>& chunks, const Loan& slots, hipStream_t s)
    {
        const size_t last = chunks.size() - 1, count = slots.count;
        const auto slot = [&](size_t k) -> const SlotPool::Slot& { return *slots.slot[k % count]; };
        hipError_t e = hipSuccess;
        size_t issued = 0;
        for (size_t taken = 0; taken < last && e == hipSuccess; ++taken) {
            for (; e == hipSuccess && issued <= last && issued < taken + count; ++issued)
                e = issued < last ? issue(chunks[issued], slot(issued), s) : copy(chunks[last], slot(last), s);
            if (e == hipSuccess) e = take(chunks[taken], slot(taken));
        }
        if (e == hipSuccess && issued <= last) e = copy(chunks[last], slot(last), s);
        const hipError_t w = hipStreamSynchronize(s);  // no copy into a slot outlives the call
        if (e == hipSuccess && w == hipSuccess) unload(chunks[last], slot(last));
        return e != hipSuccess ? e : w;
    }

    // The other threads sleep until the stream has come to the readback: the
    // runtime's waits spin, and twelve of them through a run of 2000 steps at
    // 4096^2 took 1.7 s of processor time in 0.14 s.
    static hipError_t threaded(const std::vector<Chunk>& chunks, const Loan& slots, hipStream_t s, int dev)
    {
        const size_t n = chunks.size();
        const size_t hw = std::max(1u, std::thread::hardware_concurrency());
        const size_t workers = std::min({slots.count, n, hw});
        std::atomic<int> error{(int)hipSuccess};
        std::atomic<size_t> next{0};
        size_t issued = 0;  // chunk w is worker w's first, on its way before the worker wakes
        std::mutex gate;
        std::condition_variable opened;
        bool open = false;
        auto rest = [&](size_t w, hipError_t e) {
            for (size_t k; e == hipSuccess && error.load() == (int)hipSuccess && (k = next.fetch_add(1)) < n;) {
                e = issue(chunks[k], *slots.slot[w], s);
                if (e == hipSuccess) e = take(chunks[k], *slots.slot[w]);
            }
            if (e != hipSuccess) error.store((int)e);
        };
        auto work = [&](size_t w) {
            {
                std::unique_lock<std::mutex> lock(gate);
                opened.wait(lock, [&] { return open; });
            }
            hipError_t e = hipSetDevice(dev);
            if (e == hipSuccess && w < issued) e = take(chunks[w], *slots.slot[w]);
            rest(w, e);
        };
        std::vector<std::thread> threads;
        hipError_t e = issue(chunks[0], *slots.slot[0], s);
        if (e == hipSuccess) issued = 1;
        try {
            threads.reserve(workers);
            while (e == hipSuccess && issued < workers) {
                threads.emplace_back(work, issued);
                e = issue(chunks[issued], *slots.slot[issued], s);
                if (e == hipSuccess) ++issued;
            }
        } catch (...) {  // no thread to be had: the ones that started, and this one, do the work
        }
        if (e == hipSuccess) e = hipEventSynchronize(slots.slot[0]->event);
        if (e != hipSuccess) error.store((int)e);
        next.store(issued);
        {
            std::lock_guard<std::mutex> lock(gate);
            open = true;
        }
        opened.notify_all();
        if (e == hipSuccess) unload(chunks[0], *slots.slot[0]);
        rest(0, e);
        for (std::thread& t : threads) t.join();
        const hipError_t w = hipStreamSynchronize(s);
        return error.load() != (int)hipSuccess ? (hipError_t)error.load() : w;
    }

    SlotPool* pool_ = nullptr;  // from the first readback on
};

}  // namespace lbm
