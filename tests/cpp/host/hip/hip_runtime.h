// The part of HIP that csrc/uw_rows.h and the headers under it use, for a host compiler: device functions
// become ordinary ones, and the 256 threads of a workgroup run as fibers, one at a time. An operation across
// lanes or a barrier is a meeting point: a fiber waits there until the lanes of its wave (the threads of the
// workgroup) have all come. Between meeting points the fibers run in any order, so an exchange through
// memory that lacks one of its barriers gives wrong results here.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <vector>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(n) alignas(n)

struct uint2 { uint32_t x, y; };
struct uint3 { uint32_t x, y, z; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
struct alignas(16) float4 { float x, y, z, w; };
inline uint2 make_uint2(uint32_t x, uint32_t y) { return {x, y}; }
inline uint3 make_uint3(uint32_t x, uint32_t y, uint32_t z) { return {x, y, z}; }
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }

typedef struct hip_event* hipEvent_t;
typedef struct hip_stream* hipStream_t;
typedef struct hip_graph* hipGraph_t;
typedef struct hip_graph_exec* hipGraphExec_t;
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0;

struct host_dim3 { uint32_t x = 0, y = 0, z = 0; };
inline host_dim3 threadIdx;

namespace host_block {
constexpr int kThreads = 256, kWave = 64;
struct Fiber {
    ucontext_t ctx;
    std::vector<char> stack = std::vector<char>(128 << 10);
    long met_wave = 0, met_block = 0;  // meetings it has come to
    bool done = true;
};
inline Fiber fibers[kThreads];
inline ucontext_t scheduler;
inline uint64_t mail[2][kThreads];  // exchange slots, alternating so that a fast lane overwrites no unread one
inline void (*body)(void*);
inline void* body_arg;

inline void yield() {
    const int me = int(threadIdx.x);
    swapcontext(&fibers[me].ctx, &scheduler);
}
inline void meet_wave() {
    const int me = int(threadIdx.x), w0 = me / kWave * kWave;
    const long n = ++fibers[me].met_wave;
    for (;;) {
        bool all = true;
        for (int i = w0; i < w0 + kWave; ++i) all = all && (fibers[i].done || fibers[i].met_wave >= n);
        if (all) return;
        yield();
    }
}
inline void meet_block() {
    const long n = ++fibers[threadIdx.x].met_block;
    for (;;) {
        bool all = true;
        for (const Fiber& f : fibers) all = all && (f.done || f.met_block >= n);
        if (all) return;
        yield();
    }
}
// v of every lane of the wave, as an array
inline const uint64_t* exchange(uint64_t v) {
    const int me = int(threadIdx.x);
    uint64_t* box = mail[fibers[me].met_wave & 1];
    box[me] = v;
    meet_wave();
    return box + me / kWave * kWave;
}
inline void entry() {
    body(body_arg);
    fibers[threadIdx.x].done = true;
}
// Runs body(arg) as a workgroup; seed: the order in which fibers get their turns.
inline void run(void (*f)(void*), void* arg, uint32_t seed) {
    body = f;
    body_arg = arg;
    for (Fiber& b : fibers) {
        getcontext(&b.ctx);
        b.ctx.uc_stack.ss_sp = b.stack.data();
        b.ctx.uc_stack.ss_size = b.stack.size();
        b.ctx.uc_link = &scheduler;
        b.met_wave = b.met_block = 0;
        b.done = false;
        makecontext(&b.ctx, entry, 0);
    }
    const int first = int(seed % kThreads), step = int(seed / kThreads % 128) * 2 + 1;  // odd: visits all
    for (int left = kThreads; left > 0;) {
        left = 0;
        for (int i = 0; i < kThreads; ++i) {
            const int t = (first + i * step) % kThreads;
            if (fibers[t].done) continue;
            threadIdx.x = uint32_t(t);
            swapcontext(&scheduler, &fibers[t].ctx);
            left += fibers[t].done ? 0 : 1;
        }
    }
}
}  // namespace host_block

inline void __syncthreads() { host_block::meet_block(); }
inline void __builtin_amdgcn_fence(int, const char*) {}
inline void __builtin_amdgcn_wave_barrier() { host_block::meet_wave(); }
inline int __builtin_amdgcn_readlane(int v, int lane) { return int(host_block::exchange(uint32_t(v))[lane & 63]); }
inline int __builtin_amdgcn_ds_bpermute(int at, int v) { return int(host_block::exchange(uint32_t(v))[(at >> 2) & 63]); }
inline int __builtin_amdgcn_readfirstlane(int v) { return int(host_block::exchange(uint32_t(v))[0]); }
inline bool __any(bool v) {
    const uint64_t* b = host_block::exchange(v);
    return std::any_of(b, b + 64, [](uint64_t x) { return x != 0; });
}
// row_shr:n (0x110 + n), row_bcast:15 (0x142), row_bcast:31 (0x143); lanes without a source, or in rows that
// row_mask leaves out, keep `old`
inline int __builtin_amdgcn_update_dpp(int old, int v, int ctrl, int row_mask, int, bool) {
    const uint64_t* b = host_block::exchange(uint32_t(v));
    const int lane = int(threadIdx.x & 63), row = lane >> 4;
    if (!(row_mask >> row & 1)) return old;
    if (ctrl > 0x110 && ctrl < 0x120) return (lane & 15) >= ctrl - 0x110 ? int(b[lane - (ctrl - 0x110)]) : old;
    if (ctrl == 0x142) return row > 0 ? int(b[16 * row - 1]) : old;
    if (ctrl == 0x143) return lane >= 32 ? int(b[31]) : old;
    abort();
}
inline uint32_t __builtin_amdgcn_alignbit(uint32_t hi, uint32_t lo, uint32_t s) {
    return uint32_t((uint64_t(hi) << 32 | lo) >> (s & 31u));
}
inline uint32_t __popc(uint32_t v) { return uint32_t(__builtin_popcount(v)); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return uint32_t(uint64_t(a) * b >> 32); }
inline long long __double_as_longlong(double v) { long long r; memcpy(&r, &v, 8); return r; }
inline double __longlong_as_double(long long v) { double r; memcpy(&r, &v, 8); return r; }
inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p += v; return o; }
using std::max;
using std::min;
