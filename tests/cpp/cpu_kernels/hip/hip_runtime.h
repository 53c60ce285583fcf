// A stand-in for the HIP runtime header under which g++ compiles the kernels
// of flipengine3d_amd/csrc for the host (tests/cpu_kernels.py): a workgroup's
// threads are fibers that run in turn, each until it waits at a barrier or in
// a wave exchange.  It holds what the kernels under test use and no more.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>

#define __device__
#define __host__
#define __global__
#define __constant__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))

typedef int hipError_t;
typedef void *hipStream_t;
typedef void *hipEvent_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipFuncAttributeMaxDynamicSharedMemorySize = 8 };
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void *, int, int) { return hipSuccess; }

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct int4 {
    int x, y, z, w;
};
struct float4 {
    float x, y, z, w;
};
inline int4 make_int4(int a, int b, int c, int d) { return int4{a, b, c, d}; }
inline float4 make_float4(float a, float b, float c, float d) { return float4{a, b, c, d}; }
using std::max;
using std::min;

namespace cpu {
extern dim3 thread_idx, block_idx, block_dim, grid_dim;
extern char *dynamic_lds;
extern uint64_t exchange[1024];
// Called each time a thread of a workgroup stops running (it waits or ends).
extern std::function<void()> on_yield;
void block_wait();
void wave_wait();
void launch(unsigned grid, unsigned block, size_t lds, const std::function<void()> &body);

template <class T, class From>
T wave_exchange(T v, From &&from) {
    const unsigned t = thread_idx.x;
    std::memcpy(&exchange[t], &v, sizeof(T));
    wave_wait();
    T r;
    std::memcpy(&r, &exchange[(t & ~63u) + (from(t & 63u) & 63u)], sizeof(T));
    wave_wait();
    return r;
}
}  // namespace cpu
#define threadIdx cpu::thread_idx
#define blockIdx cpu::block_idx
#define blockDim cpu::block_dim
#define gridDim cpu::grid_dim

inline void __syncthreads() { cpu::block_wait(); }
inline int __syncthreads_or(int v) {
    static int any;
    __syncthreads();
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    if (v) any = 1;
    __syncthreads();
    return any;
}
template <class T>
T __shfl_xor(T v, int mask, int = 64) {
    return cpu::wave_exchange(v, [=](unsigned l) { return l ^ (unsigned)mask; });
}
template <class T>
T __shfl(T v, int src, int = 64) {
    return cpu::wave_exchange(v, [=](unsigned) { return (unsigned)src; });
}
template <class T>
T __shfl_up(T v, int off, int = 64) {
    return cpu::wave_exchange(v, [=](unsigned l) { return l >= (unsigned)off ? l - (unsigned)off : l; });
}
inline unsigned long long __ballot(int v) {
    unsigned long long m = 0;
    for (int q = 0; q < 64; q++) m |= (unsigned long long)(__shfl(v, q) != 0) << q;
    return m;
}
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
template <class T, class U>
T atomicAdd(T *p, U v) {
    T o = *p;
    *p += v;
    return o;
}
template <class T, class U>
T atomicOr(T *p, U v) {
    T o = *p;
    *p |= v;
    return o;
}
template <class T>
T bits_as(uint32_t u) {
    T v;
    std::memcpy(&v, &u, 4);
    return v;
}
inline uint32_t __float_as_uint(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}
inline float __uint_as_float(uint32_t u) { return bits_as<float>(u); }
inline int __float_as_int(float f) { return (int)__float_as_uint(f); }
inline float __int_as_float(int u) { return bits_as<float>((uint32_t)u); }
