// HIP on the CPU, for tests that run kernels and the host code that plans and
// launches them without a device: every thread of a workgroup is a context of
// its own, switched at barriers and wave operations; workgroups run one after
// another.  Device memory starts with hipcpu::stale, repeated; a barrier that some threads of
// its workgroup have left behind ends the program, and hooks let a test act where
// another workgroup would (hipcpu::before_wave) or fail an allocation
// (hipcpu::memory_left).  Captured launches run when their graph does.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <functional>
#include <map>
#include <memory>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) alignas(n)

struct int2 { int x, y; };
struct uint2 { uint32_t x, y; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
struct alignas(16) double2 { double x, y; };
struct alignas(16) double4 { double x, y, z, w; };
struct dim3 {
    uint32_t x, y, z;
    dim3(uint32_t a = 1, uint32_t b = 1, uint32_t c = 1) : x(a), y(b), z(c) {}
};
inline int2 make_int2(int x, int y) { return {x, y}; }
inline uint2 make_uint2(uint32_t x, uint32_t y) { return {x, y}; }
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }
inline double2 make_double2(double x, double y) { return {x, y}; }
inline double4 make_double4(double x, double y, double z, double w) { return {x, y, z, w}; }

namespace hipcpu {

enum State { READY, WAVE_OP, BARRIER, DONE };
struct Thread {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    dim3 tid;
    State state = DONE;
    uint64_t val = 0;
};
constexpr size_t STACK = 64 << 10;
inline std::vector<std::unique_ptr<Thread>> pool;
inline Thread *cur = nullptr;
inline ucontext_t back;
inline dim3 block_idx, block_dim, grid_dim;
inline uint64_t snap[16][64];  // values of a wave's last operation
inline uint64_t arrived[16];   // lanes that took part in it
inline bool any = false, any_out = false;
inline const std::function<void()> *body = nullptr;
// called before the given wave of a workgroup first runs: kernel, workgroup, wave
inline std::function<void(const void *, uint32_t, uint32_t)> before_wave;
inline uint64_t barriers = 0;  // passed by workgroups so far
// called before a launch: kernel, its first argument
inline std::function<void(const void *, const void *)> before_launch;

[[noreturn]] inline void die(const char *what)
{
    fprintf(stderr, "hipcpu: %s (workgroup %u)\n", what, block_idx.x);
    exit(3);
}

inline void entry()
{
    (*body)();
    cur->state = DONE;
    swapcontext(&cur->ctx, &back);
}

inline void yield(State s)
{
    cur->state = s;
    swapcontext(&cur->ctx, &back);
}

inline void run_block(const void *kernel, uint32_t n)
{
    while (pool.size() < n) {
        pool.emplace_back(new Thread);
        pool.back()->stack.reset(new char[STACK]);
    }
    for (uint32_t i = 0; i < n; ++i) {
        Thread &t = *pool[i];
        getcontext(&t.ctx);
        t.ctx.uc_stack.ss_sp = t.stack.get();
        t.ctx.uc_stack.ss_size = STACK;
        t.ctx.uc_link = nullptr;
        makecontext(&t.ctx, entry, 0);
        t.tid = dim3(i, 0, 0);
        t.state = READY;
    }
    const uint32_t waves = (n + 63) / 64;
    bool first = true;
    for (uint64_t rounds = 0;; ++rounds) {
        if (rounds > 1000000)
            die("a workgroup that does not end");
        uint32_t done = 0;
        for (uint32_t w = 0; w < waves; ++w) {
            if (first && before_wave)
                before_wave(kernel, block_idx.x, w);
            const uint32_t a = w * 64, b = a + 64 < n ? a + 64 : n;
            for (bool more = true; more;) {
                for (uint32_t i = a; i < b; ++i)
                    if (pool[i]->state == READY) {
                        cur = pool[i].get();
                        swapcontext(&back, &cur->ctx);
                    }
                more = false;
                arrived[w] = 0;
                for (uint32_t i = a; i < b; ++i)
                    if (pool[i]->state == WAVE_OP) {
                        snap[w][i - a] = pool[i]->val;
                        arrived[w] |= 1ull << (i - a);
                        pool[i]->state = READY;
                        more = true;
                    }
            }
            for (uint32_t i = a; i < b; ++i)
                done += pool[i]->state == DONE;
        }
        first = false;
        if (done == n)
            return;
        if (done)
            die("a barrier that some threads left behind");
        ++barriers;
        any_out = any;
        any = false;
        for (uint32_t i = 0; i < n; ++i)
            pool[i]->state = READY;
    }
}

struct Graph {
    std::vector<std::function<void()>> nodes;
};
inline Graph *capture = nullptr;
inline uint64_t graph_launches = 0;

template <class T, class... A> const void *first_of(const T &t, const A &...) { return &t; }

template <class... P, class... A>
void launch(void (*k)(P...), dim3 g, dim3 b, A... a)
{
    const std::function<void()> run = [=]() {
        if (before_launch)
            before_launch((const void *)k, first_of(a...));
        const std::function<void()> f = [=]() { k(a...); };
        body = &f;
        grid_dim = g;
        block_dim = b;
        for (uint32_t y = 0; y < g.y; ++y)
            for (uint32_t x = 0; x < g.x; ++x) {
                block_idx = dim3(x, y, 0);
                run_block((const void *)k, b.x);
            }
    };
    if (capture)
        capture->nodes.push_back(run);
    else
        run();
}

// bytes that further allocations may take (freed ones come back)
inline uint64_t memory_left = ~0ull;
inline uint64_t largest = 0;  // allocation asked for
inline std::map<void *, uint64_t> sizes;
// what device memory holds before it is written
inline std::vector<unsigned char> stale{0xA5};

inline uint64_t wave_op(uint64_t v)
{
    cur->val = v;
    yield(WAVE_OP);
    return v;
}
template <class T> T from_lane(uint32_t src, T own)
{
    const uint32_t w = cur->tid.x >> 6;
    if (src > 63u || !((arrived[w] >> src) & 1ull))
        return own;
    T v;
    memcpy(&v, &snap[w][src], sizeof v);
    return v;
}
template <class T> T shuffle(T v, uint32_t src)
{
    uint64_t u = 0;
    memcpy(&u, &v, sizeof v);
    wave_op(u);
    return from_lane(src, v);
}

}  // namespace hipcpu

#define threadIdx (hipcpu::cur->tid)
#define blockIdx hipcpu::block_idx
#define blockDim hipcpu::block_dim
#define gridDim hipcpu::grid_dim
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) hipcpu::launch(k, grid, block, __VA_ARGS__)

inline uint32_t __lane_id() { return threadIdx.x & 63u; }
inline void __syncthreads() { hipcpu::yield(hipcpu::BARRIER); }
inline int __syncthreads_or(int p)
{
    hipcpu::any = hipcpu::any || p;
    hipcpu::yield(hipcpu::BARRIER);
    return hipcpu::any_out;
}
inline void __threadfence() {}
inline void __builtin_amdgcn_wave_barrier() { hipcpu::wave_op(0); }
inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v) { return v; }  // of values that are uniform
template <class T> T __shfl(T v, int src, int) { return hipcpu::shuffle(v, (uint32_t)src); }
template <class T> T __shfl_up(T v, int o, int) { return hipcpu::shuffle(v, __lane_id() - (uint32_t)o); }
template <class T> T __shfl_xor(T v, int o, int) { return hipcpu::shuffle(v, __lane_id() ^ (uint32_t)o); }
inline unsigned long long __ballot(int p)
{
    hipcpu::wave_op(p != 0);
    const uint32_t w = threadIdx.x >> 6;
    unsigned long long m = 0;
    for (uint32_t l = 0; l < 64; ++l)
        if (((hipcpu::arrived[w] >> l) & 1ull) && hipcpu::snap[w][l])
            m |= 1ull << l;
    return m;
}
inline const char *__builtin_amdgcn_make_buffer_rsrc(void *p, int, uint32_t, uint32_t) { return (const char *)p; }
inline uint32_t __builtin_amdgcn_raw_buffer_load_b32(const char *p, uint32_t at, uint32_t, int)
{
    uint32_t v;
    memcpy(&v, p + at, 4);
    return v;
}
template <class T> T min(T a, T b) { return b < a ? b : a; }
template <class T> T max(T a, T b) { return a < b ? b : a; }
template <class T> T atomicAdd(T *p, T v) { const T o = *p; *p = o + v; return o; }
template <class T> T atomicOr(T *p, T v) { const T o = *p; *p = o | v; return o; }
template <class T> T atomicMin(T *p, T v) { const T o = *p; *p = v < o ? v : o; return o; }
template <class T> T atomicExch(T *p, T v) { const T o = *p; *p = v; return o; }
inline int __popc(uint32_t v) { return __builtin_popcount(v); }
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline long long __double_as_longlong(double v) { long long r; memcpy(&r, &v, 8); return r; }
inline double __hiloint2double(int hi, int lo)
{
    const uint64_t b = (uint64_t)(uint32_t)hi << 32 | (uint32_t)lo;
    double v;
    memcpy(&v, &b, 8);
    return v;
}
inline double __dadd_rn(double a, double b) { return a + b; }
inline double __dsub_rn(double a, double b) { return a - b; }
inline double __dmul_rn(double a, double b) { return a * b; }

// ----------------------------------------------------------- host calls --

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum { hipStreamCaptureModeThreadLocal, hipFuncAttributeMaxDynamicSharedMemorySize };
typedef void *hipStream_t;
typedef void *hipEvent_t;
typedef hipcpu::Graph *hipGraph_t;
typedef hipcpu::Graph *hipGraphExec_t;

inline hipError_t hipMalloc(void **p, uint64_t n)
{
    *p = nullptr;
    hipcpu::largest = n > hipcpu::largest ? n : hipcpu::largest;
    if (n > hipcpu::memory_left)
        return hipErrorOutOfMemory;
    *p = malloc(n);
    for (uint64_t i = 0; i < n; i += hipcpu::stale.size())
        memcpy((char *)*p + i, hipcpu::stale.data(),
               n - i < hipcpu::stale.size() ? n - i : hipcpu::stale.size());
    hipcpu::sizes[*p] = n;
    if (hipcpu::memory_left != ~0ull)
        hipcpu::memory_left -= n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p)
{
    if (hipcpu::memory_left != ~0ull)
        hipcpu::memory_left += hipcpu::sizes[p];
    free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, uint64_t n, unsigned)
{
    *p = malloc(n);
    memset(*p, 0xA5, n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipMemcpy(void *d, const void *s, uint64_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, uint64_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 0.f; return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void *, int, int) { return hipSuccess; }
inline hipError_t hipStreamBeginCapture(hipStream_t, int) { hipcpu::capture = new hipcpu::Graph; return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = hipcpu::capture; hipcpu::capture = nullptr; return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, void *, void *, int) { *e = new hipcpu::Graph(*g); return hipSuccess; }
inline hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t g) { delete g; return hipSuccess; }
inline hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t)
{
    ++hipcpu::graph_launches;
    for (auto &f : g->nodes)
        f();
    return hipSuccess;
}
