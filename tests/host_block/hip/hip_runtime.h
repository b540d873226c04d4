// A thread block of a HIP kernel on the CPU, for tests of the order in which
// its threads use LDS.
//
// The kernel sources are compiled for the host with this header in place of
// HIP's.  Every thread of a block is a fiber, LDS is static memory, and a
// fiber runs without interruption from one barrier to the next: `order` says
// which threads go first.  A kernel whose barriers order every access to LDS
// gives the same bits in every order; where one thread may write what another
// has still to read, some order shows it.  One block runs at a time.  The
// operations across lanes (DPP moves, ballots) are not modelled: a kernel that
// needs them ends the program.
#pragma once

#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
struct double2 { double x, y; };
inline double2 make_double2(double x, double y) { return {x, y}; }
using hipError_t = int;
using hipStream_t = void *;
enum { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice };
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(to, from, n);
    return hipSuccess;
}

static dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace host_block {

enum class Order { ascending, descending, waves_descending };
static Order order = Order::ascending;

struct Fiber {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    bool done = false;
};
static std::vector<Fiber> fibers;
static ucontext_t scheduler;
static unsigned running = 0;
static std::function<void()> body;

inline void barrier() { swapcontext(&fibers[running].ctx, &scheduler); }

inline void entry()
{
    body();
    fibers[running].done = true;
    swapcontext(&fibers[running].ctx, &scheduler);
}

inline void run_block(unsigned threads)
{
    constexpr size_t kStack = 256 << 10;
    fibers.resize(std::max<size_t>(fibers.size(), threads));
    for (unsigned t = 0; t < threads; ++t) {
        Fiber &f = fibers[t];
        if (!f.stack) f.stack.reset(new char[kStack]);
        f.done = false;
        getcontext(&f.ctx);
        f.ctx.uc_stack.ss_sp = f.stack.get();
        f.ctx.uc_stack.ss_size = kStack;
        f.ctx.uc_link = nullptr;
        makecontext(&f.ctx, entry, 0);
    }
    for (unsigned left = threads; left > 0;) {
        for (unsigned i = 0; i < threads; ++i) {
            unsigned t = i;
            if (order == Order::descending) t = threads - 1 - i;
            if (order == Order::waves_descending) {
                t = (threads / 64 - 1 - i / 64) * 64 + i % 64;
            }
            if (fibers[t].done) continue;
            running = t;
            threadIdx = dim3(t, 0, 0);
            swapcontext(&scheduler, &fibers[t].ctx);
            left -= fibers[t].done ? 1 : 0;
        }
    }
}

template <class K, class... A>
void launch(K kernel, dim3 grid, dim3 block, A... args)
{
    gridDim = grid;
    blockDim = block;
    body = [=] { kernel(args...); };
    for (unsigned b = 0; b < grid.x; ++b) {
        blockIdx = dim3(b, 0, 0);
        run_block(block.x);
    }
}

[[noreturn]] inline int not_modelled()
{
    std::fprintf(stderr, "an operation across lanes\n");
    std::abort();
}

}  // namespace host_block

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n)
#define __syncthreads() host_block::barrier()
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    host_block::launch(kernel, grid, block, __VA_ARGS__)
// the kernels' asm statements are empty: they only hold the compiler back
#define volatile(...)
#define asm

#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt(double(x)))
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(float(x)))
#define __builtin_amdgcn_sqrtf(x) std::sqrt(float(x))
#define __builtin_amdgcn_exp2f(x) std::exp2(float(x))
#define __builtin_amdgcn_logf(x) std::log2(float(x))
#define __builtin_amdgcn_s_setprio(x)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_readfirstlane(x) (x)  // of a value every lane holds
#define __builtin_amdgcn_wave_barrier() host_block::not_modelled()
#define __builtin_amdgcn_update_dpp(...) host_block::not_modelled()
#define __builtin_amdgcn_readlane(...) host_block::not_modelled()
#define __ballot(x) ((unsigned long long)host_block::not_modelled())
#define __popcll(x) __builtin_popcountll(x)

inline unsigned __umulhi(unsigned a, unsigned b)
{
    return unsigned((unsigned long long)a * b >> 32);
}
inline long long __double_as_longlong(double v)
{
    long long b;
    std::memcpy(&b, &v, 8);
    return b;
}
inline double __longlong_as_double(long long b)
{
    double v;
    std::memcpy(&v, &b, 8);
    return v;
}
inline int atomicCAS(int *p, int expected, int v)
{
    const int old = *p;
    if (old == expected) *p = v;
    return old;
}
inline unsigned long long atomicMin(unsigned long long *p, unsigned long long v)
{
    const unsigned long long old = *p;
    *p = std::min(old, v);
    return old;
}
using std::fabs;
using std::max;
using std::min;
using std::sqrt;
