// What a kernel source needs to run on the CPU, in place of the HIP header of that name: a group's threads are contexts that take turns
// between barriers, a raw buffer checks its range as the hardware does. Slow; for checks of where kernels read and write.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __noinline__ __attribute__((noinline))
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n) __attribute__((aligned(n)))
#define amdgpu_waves_per_eu(...) unused
#define asm(...)  // (values that pass through one are not looked at here)
using std::max;
using std::min;

typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0;
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return ""; }
template <typename T>
hipError_t hipGetSymbolAddress(void** p, const T& symbol) { *p = (void*)&symbol; return hipSuccess; }
#define HIP_SYMBOL(x) x
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct int4 { int x, y, z, w; };
struct float4 { float x, y, z, w; };
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }

namespace host {
struct index { unsigned x, y, z; };
inline index thread, block, threads, blocks;
struct context {
    ucontext_t at;
    bool done;
    int value;
};
inline std::vector<context> group;
inline std::vector<std::vector<char>> stacks;
inline ucontext_t scheduler;
inline int current;
inline const std::function<void()>* body;

inline void barrier() { swapcontext(&group[current].at, &scheduler); }
inline void enter() {
    (*body)();
    group[current].done = true;
    swapcontext(&group[current].at, &scheduler);
}
// Every thread runs to the next barrier, or its end, before any goes on behind it.
inline void launch(dim3 g, dim3 b, const std::function<void()>& f) {
    const int n = (int)(b.x * b.y * b.z);
    body = &f;
    group.resize(n);
    stacks.resize(n);
    blocks = {g.x, g.y, g.z};
    threads = {b.x, b.y, b.z};
    for (unsigned i = 0; i < g.x * g.y * g.z; ++i) {
        block = {i % g.x, i / g.x % g.y, i / g.x / g.y};
        for (int t = 0; t < n; ++t) {
            stacks[t].resize(65536);
            group[t].done = false;
            getcontext(&group[t].at);
            group[t].at.uc_stack.ss_sp = stacks[t].data();
            group[t].at.uc_stack.ss_size = stacks[t].size();
            makecontext(&group[t].at, enter, 0);
        }
        for (bool left = true; left;) {
            left = false;
            for (current = 0; current < n; ++current) {
                if (group[current].done) continue;
                thread = {current % b.x, current / b.x % b.y, current / b.x / b.y};
                swapcontext(&scheduler, &group[current].at);
                left = left || !group[current].done;
            }
        }
    }
}
// Another lane's value; every thread of the group asks at once.
template <typename T>
T of_lane(T v, int lane) {
    static_assert(sizeof(T) == 4, "a register");
    memcpy(&group[current].value, &v, 4);
    barrier();
    memcpy(&v, &group[(current & ~63) + lane].value, 4);
    barrier();
    return v;
}
}  // namespace host
#define threadIdx host::thread
#define blockIdx host::block
#define blockDim host::threads
#define gridDim host::blocks
inline void __syncthreads() { host::barrier(); }
template <typename T>
T __shfl_xor(T v, int mask, int = 64) { return host::of_lane(v, (host::current & 63) ^ mask); }
template <typename T>
T __shfl_down(T v, int by, int = 64) { return host::of_lane(v, std::min((host::current & 63) + by, 63)); }
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) host::launch(grid, block, [&] { (kernel)(__VA_ARGS__); })

struct host_buffer {
    char* at;
    unsigned bytes;
};
#define __amdgpu_buffer_rsrc_t host_buffer
template <int WORDS>
using host_words = unsigned __attribute__((ext_vector_type(WORDS)));
template <typename V>
V host_load(host_buffer r, unsigned lane, unsigned scalar) {
    V v = {};
    for (size_t i = 0; i < sizeof(V); i += 4)
        if ((size_t)lane + scalar + i + 4 <= r.bytes) memcpy((char*)&v + i, r.at + lane + scalar + i, 4);
    return v;
}
template <typename V>
void host_store(V v, host_buffer r, unsigned lane, unsigned scalar) {
    for (size_t i = 0; i < sizeof(V); i += 4)
        if ((size_t)lane + scalar + i + 4 <= r.bytes) memcpy(r.at + lane + scalar + i, (char*)&v + i, 4);
}
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, n, word3) host_buffer{(char*)(p), (unsigned)(n)}
#define __builtin_amdgcn_raw_buffer_load_b128(r, lane, scalar, aux) host_load<host_words<4>>(r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_load_b64(r, lane, scalar, aux) host_load<host_words<2>>(r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_load_b32(r, lane, scalar, aux) host_load<unsigned>(r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_store_b128(v, r, lane, scalar, aux) host_store(v, r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_store_b64(v, r, lane, scalar, aux) host_store(v, r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_store_b32(v, r, lane, scalar, aux) host_store(v, r, lane, scalar)
#define __builtin_amdgcn_fmed3f(a, b, c) fmaxf(fminf(fmaxf(a, b), c), fminf(a, b))
#define __builtin_amdgcn_mov_dpp(v, control, rows, banks, bound) (v)
struct host_pair {
    unsigned v[2];
    unsigned operator[](int i) const { return v[i]; }
};
#define __builtin_amdgcn_permlane32_swap(a, b, f, c) (host_pair{{a, b}})
