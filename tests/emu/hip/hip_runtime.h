// Stand-in for the HIP runtime header: the names that the cell kernels use, for
// g++.  Lanes of a wave are coroutines of one thread (rt.cpp); an operation
// across lanes waits until every lane of the wave has come to it.
#pragma once

#include <float.h>
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __host__
#define __global__ [[maybe_unused]] static
#define __forceinline__ inline
#define __noinline__
#define __shared__ static
#define __launch_bounds__(...)

struct alignas(16) float4 {
    float x, y, z, w;
};
struct alignas(8) float2 {
    float x, y;
};
struct alignas(8) uint2 {
    unsigned x, y;
};
inline float4 make_float4(float x, float y, float z, float w) { return float4{x, y, z, w}; }
inline float2 make_float2(float x, float y) { return float2{x, y}; }

typedef int hipError_t;
typedef void *hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
inline hipError_t hipGetLastError() { return hipSuccess; }
#define hipLaunchKernelGGL(...) ((void)0)

namespace emu {
extern int lane;  // the lane that runs now
enum Op : int { kBallot = 1, kShuffle, kShuffleXor, kDpp, kReadLane, kReadFirst, kFence };
// every lane of the wave brings a value; returns the values, by lane
const uint32_t *meet(Op op, int arg, uint32_t x);
int lanes();
uint64_t ballot(bool p);
uint32_t dpp(uint32_t x, int ctrl);
void fence();
void atomic_at(const void *p, int bytes);  // the lane's next access there is an atomic one
struct Idx {
    unsigned x, y, z;
};
inline Idx tid() { return Idx{(unsigned)lane, 0u, 0u}; }
inline uint32_t bits(float x) {
    uint32_t u;
    memcpy(&u, &x, 4);
    return u;
}
inline float flt(uint32_t u) {
    float x;
    memcpy(&x, &u, 4);
    return x;
}
inline uint32_t shfl(uint32_t x, int src, int width) {
    return meet(kShuffle, width, x)[(lane & ~(width - 1)) + (src & (width - 1))];
}
}  // namespace emu

#define threadIdx emu::tid()
#define blockIdx (emu::Idx{0u, 0u, 0u})
#define blockDim (emu::Idx{64u, 1u, 1u})
#define gridDim (emu::Idx{1u, 1u, 1u})
inline void __syncthreads() {}
inline uint64_t clock64() { return 0; }

inline uint64_t __ballot(bool p) { return emu::ballot(p); }
inline int __shfl(int x, int src, int width = 64) { return (int)emu::shfl((uint32_t)x, src, width); }
inline float __shfl(float x, int src, int width = 64) { return emu::flt(emu::shfl(emu::bits(x), src, width)); }
inline uint32_t __shfl_xor(uint32_t x, int m) { return emu::meet(emu::kShuffleXor, m, x)[emu::lane ^ m]; }
inline uint32_t __float_as_uint(float x) { return emu::bits(x); }
inline int __float_as_int(float x) { return (int)emu::bits(x); }
inline float __uint_as_float(uint32_t u) { return emu::flt(u); }
inline float __int_as_float(int u) { return emu::flt((uint32_t)u); }
inline int __popc(uint32_t x) { return __builtin_popcount(x); }
inline int __popcll(uint64_t x) { return __builtin_popcountll(x); }
template <class T>
inline T min(T a, T b) {
    return b < a ? b : a;
}
template <class T>
inline T max(T a, T b) {
    return a < b ? b : a;
}
template <class T, class U>
inline T atomicAdd(T *p, U v) {
    emu::atomic_at(p, sizeof(T));
    const T o = *p;
    *p = (T)(o + (T)v);
    return o;
}
template <class T, class U>
inline T atomicOr(T *p, U v) {
    emu::atomic_at(p, sizeof(T));
    const T o = *p;
    *p = (T)(o | (T)v);
    return o;
}
template <class T, class U>
inline T atomicMax(T *p, U v) {
    emu::atomic_at(p, sizeof(T));
    const T o = *p;
    *p = o < (T)v ? (T)v : o;
    return o;
}

#define __HIP_MEMORY_SCOPE_WAVEFRONT 0
#define __hip_atomic_load(p, order, scope) (*(p))
#define __builtin_amdgcn_fence(...) emu::fence()
#define __builtin_amdgcn_readlane(x, l) ((int)emu::meet(emu::kReadLane, 0, (uint32_t)(x))[l])
#define __builtin_amdgcn_readfirstlane(x) ((int)emu::meet(emu::kReadFirst, 0, (uint32_t)(x))[0])
#define __builtin_amdgcn_update_dpp(old, x, c, rows, banks, bound) ((int)emu::dpp((uint32_t)(x), c))
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
inline float __builtin_amdgcn_fmed3f_(float a, float b, float c) { return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c)); }
#define __builtin_amdgcn_fmed3f __builtin_amdgcn_fmed3f_
// an empty asm statement with a register class of the GPU
#define asm
#define volatile(...)
