// A block of threads on the CPU, for host tests that compile kernels of
// openstaple_amd/csrc as plain C++ (clang++, with this folder before the HIP
// headers).  Every thread is a fiber that runs until it waits for its wave
// (shuffles, ballots) or its block (__syncthreads); blocks run one after the
// other.  Only what those kernels use is here.
#pragma once

#include <math.h>
#include <setjmp.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <vector>

#define __device__
#define __host__
#define __global__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n) alignas(n)
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x)
#define __clzll(x) __builtin_clzll(x)

struct alignas(16) double2 {
    double x, y;
};
struct alignas(8) float2 {
    float x, y;
};
inline double2 make_double2(double x, double y) { return double2{x, y}; }
inline float2 make_float2(float x, float y) { return float2{x, y}; }
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
typedef struct ihipStream_t* hipStream_t;
typedef int hipError_t;
using std::min;

static dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace hostblock {

struct Fiber {
    jmp_buf env;
    ucontext_t ctx;
    bool started = false, done = false;
    std::vector<char> stack;
};
static std::vector<Fiber> fibers;
static std::function<void()> body;
static jmp_buf scheduler;
static int cur, live, block_n, block_gen, wave_n[16], wave_gen[16];
static double wave_val[16][64];
static int wave_bit[16][64];

inline void yield() {
    if (_setjmp(fibers[cur].env) == 0) _longjmp(scheduler, 1);
}
inline void wave_wait() {
    const int w = cur >> 6, gen = wave_gen[w];
    if (++wave_n[w] == 64) {
        wave_n[w] = 0;
        wave_gen[w]++;
    } else {
        while (wave_gen[w] == gen) yield();
    }
}
inline void block_wait() {
    const int gen = block_gen;
    if (++block_n == live) {
        block_n = 0;
        block_gen++;
    } else {
        while (block_gen == gen) yield();
    }
}
inline void entry() {
    body();
    fibers[cur].done = true;
    _longjmp(scheduler, 1);
}

// f() by every thread of every block of the grid
template <class F>
void launch(dim3 grid, int threads, F f) {
    body = f;
    gridDim = grid;
    blockDim = dim3(threads);
    if ((int)fibers.size() < threads) fibers = std::vector<Fiber>(threads);
    for (unsigned by = 0; by < grid.y; by++)
        for (unsigned bx = 0; bx < grid.x; bx++) {
            blockIdx = dim3(bx, by);
            block_n = 0;
            live = threads;
            memset(wave_n, 0, sizeof wave_n);
            for (int t = 0; t < threads; t++) {
                Fiber& b = fibers[t];
                b.started = b.done = false;
                if (b.stack.empty()) b.stack.resize(64 * 1024);
                getcontext(&b.ctx);
                b.ctx.uc_stack.ss_sp = b.stack.data();
                b.ctx.uc_stack.ss_size = b.stack.size();
                b.ctx.uc_link = nullptr;
                makecontext(&b.ctx, entry, 0);
            }
            for (long pass = 0; live > 0; pass++) {
                if (pass > 100000) {
                    fprintf(stderr, "a wait that never ends\n");
                    abort();
                }
                for (int t = 0; t < threads; t++) {
                    Fiber& b = fibers[t];
                    if (b.done) continue;
                    cur = t;
                    threadIdx = dim3(t, 0, 0);
                    if (_setjmp(scheduler) == 0) {
                        if (b.started) _longjmp(b.env, 1);
                        b.started = true;
                        setcontext(&b.ctx);
                    }
                    if (fibers[cur].done && --live > 0 && block_n == live) {
                        block_n = 0;
                        block_gen++;
                    }
                }
            }
        }
}

}  // namespace hostblock

inline void __syncthreads() { hostblock::block_wait(); }
inline double __shfl_xor(double v, int off, int) {
    using namespace hostblock;
    const int w = cur >> 6, l = cur & 63;
    wave_val[w][l] = v;
    wave_wait();
    const double r = wave_val[w][l ^ off];
    wave_wait();
    return r;
}
inline unsigned long long __ballot(int p) {
    using namespace hostblock;
    const int w = cur >> 6;
    wave_bit[w][cur & 63] = p != 0;
    wave_wait();
    unsigned long long m = 0;
    for (int l = 0; l < 64; l++) m |= (unsigned long long)wave_bit[w][l] << l;
    wave_wait();
    return m;
}
