// Enough of the device language to run a tile kernel's body on the CPU: one
// block at a time, its threads as fibers that change at __syncthreads().
#pragma once

#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <memory>
#include <vector>

#if defined(__has_feature)
#if __has_feature(address_sanitizer)
#include <sanitizer/common_interface_defs.h>
#define EMU_ASAN 1
#endif
#endif

#define __global__
#define __host__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static

struct Dim3 {
    unsigned x = 0, y = 0, z = 0;
};
inline Dim3 threadIdx, blockIdx, gridDim, blockDim;
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1 };
using hipStream_t = void*;
inline hipError_t hipGetLastError() { return hipSuccess; }
struct dim3 {
    unsigned x;
    dim3(unsigned v) : x(v) {}
};
#define hipLaunchKernelGGL(...) abort()

struct float4 { float x, y, z, w; };
struct float2 { float x, y; };
struct uint2 { unsigned x, y; };
struct uint4 { unsigned x, y, z, w; };
inline float4 make_float4(float a, float b, float c, float d) { return {a, b, c, d}; }
inline uint2 make_uint2(unsigned a, unsigned b) { return {a, b}; }

inline int min(int a, int b) { return a < b ? a : b; }

namespace emu {
inline int any_mode = 0;  // what __any answers a lane: 0 its own predicate, 1 always true

// Runs `body` once per thread of a block of n; `backwards` takes the threads in
// the other order, which a missing barrier shows.  Returns false if the threads
// did not all come to the same barriers.
class Block {
public:
    bool run(unsigned n, bool backwards, const std::function<void()>& body)
    {
        if (fibers_.size() != n) {
            fibers_.clear();
            for (unsigned k = 0; k < n; ++k) fibers_.push_back(std::make_unique<Fiber>());
        }
        self() = this;
        body_ = &body;
        for (auto& f : fibers_) {
            getcontext(&f->ctx);
            f->ctx.uc_stack.ss_sp = f->stack.data();
            f->ctx.uc_stack.ss_size = f->stack.size();
            f->ctx.uc_link = nullptr;
            makecontext(&f->ctx, &Block::entry, 0);
            f->done = false;
        }
        for (;;) {
            unsigned waiting = 0, ended = 0;
            for (unsigned k = 0; k < n; ++k) {
                const unsigned t = backwards ? n - 1 - k : k;
                cur_ = fibers_[t].get();
                if (cur_->done) return false;
                threadIdx.x = t;
                enter(*cur_);
                ++(cur_->done ? ended : waiting);
            }
            if (ended == n) return true;
            if (waiting != n) return false;
        }
    }
    void barrier() { leave(false); }
    static Block*& self()
    {
        static Block* b = nullptr;
        return b;
    }

private:
    struct Fiber {
        ucontext_t ctx;
        std::vector<char> stack = std::vector<char>(1 << 16);
        bool done = false;
        void* fake = nullptr;
    };
    static void entry()
    {
        Block& b = *self();
#ifdef EMU_ASAN
        __sanitizer_finish_switch_fiber(nullptr, &b.main_bottom_, &b.main_size_);
#endif
        (*b.body_)();
        b.cur_->done = true;
        b.leave(true);
    }
    void enter(Fiber& f)
    {
#ifdef EMU_ASAN
        void* fake;
        __sanitizer_start_switch_fiber(&fake, f.stack.data(), f.stack.size());
        swapcontext(&main_, &f.ctx);
        __sanitizer_finish_switch_fiber(fake, nullptr, nullptr);
#else
        swapcontext(&main_, &f.ctx);
#endif
    }
    void leave(bool last)
    {
        Fiber& f = *cur_;
#ifdef EMU_ASAN
        __sanitizer_start_switch_fiber(last ? nullptr : &f.fake, main_bottom_, main_size_);
        swapcontext(&f.ctx, &main_);
        __sanitizer_finish_switch_fiber(f.fake, &main_bottom_, &main_size_);
#else
        (void)last;
        swapcontext(&f.ctx, &main_);
#endif
    }
    ucontext_t main_;
    std::vector<std::unique_ptr<Fiber>> fibers_;
    Fiber* cur_ = nullptr;
    const std::function<void()>* body_ = nullptr;
    const void* main_bottom_ = nullptr;
    size_t main_size_ = 0;
};
}  // namespace emu

inline void __syncthreads() { emu::Block::self()->barrier(); }
inline int __any(int p) { return emu::any_mode ? 1 : p; }
inline unsigned __umul24(unsigned a, unsigned b)
{
    if (a >> 24 || b >> 24) abort();  // the device multiplies 24 bits
    return a * b;
}
inline double __shfl_xor(double v, int, int = 64) { return v; }

#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_alignbit(hi, lo, s) ((uint32_t)(((((uint64_t)(hi)) << 32) | (uint32_t)(lo)) >> ((s) & 31)))
#define __builtin_amdgcn_sbfe(v, bit, n) (((int)((uint32_t)(v) << (32 - (n) - (bit)))) >> (32 - (n)))
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, i, j, k) (c)
#define __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, i, j, k) (c)
typedef _Float16 emu_f16x2 __attribute__((ext_vector_type(2)));
#define __builtin_amdgcn_cvt_pkrtz(a, b) (emu_f16x2{(_Float16)(a), (_Float16)(b)})
