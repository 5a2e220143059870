// Reductions and scans over a row (16 lanes) of a wave.
#pragma once

#include "pg_common.hpp"

namespace pg {

// Row (16-lane) reductions and scans on the data-parallel-primitive path of
// the VALU: no LDS round trip, unlike ds_bpermute shuffles.
constexpr int kDppXor1 = 0xB1;   // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;   // quad_perm [2, 3, 0, 1]
constexpr int kDppRor4 = 0x124;  // row_ror:4
constexpr int kDppRor8 = 0x128;  // row_ror:8
constexpr int kDppLast = 0x15F;  // row_newbcast:15
constexpr int kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118;  // row_shr:n

template <int C>
__device__ __forceinline__ int dpp(int x) {
    return __builtin_amdgcn_update_dpp(0, x, C, 0xF, 0xF, true);  // lanes shifted in from outside the row read 0
}
// Float minima and maxima over a row through an order-preserving integer
// key (sign-magnitude bits turned into two's complement): each step is one
// integer min or max with the DPP operand folded in, where fminf/fmaxf of a
// shuffled value would add two NaN-quieting instructions per step.  The
// values reduced here are never NaN (+inf is, and orders above every finite
// value; -0 orders just below +0).
__device__ __forceinline__ int f2ord(float x) {
    const int b = __float_as_int(x);
    return b ^ ((b >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float ord2f(int o) { return __int_as_float(o ^ ((o >> 31) & 0x7fffffff)); }
__device__ __forceinline__ float row_min(float x) {
    int o = f2ord(x);
    o = min(o, dpp<kDppXor1>(o));
    o = min(o, dpp<kDppXor2>(o));
    o = min(o, dpp<kDppRor4>(o));
    return ord2f(min(o, dpp<kDppRor8>(o)));
}
__device__ __forceinline__ float row_max(float x) {
    int o = f2ord(x);
    o = max(o, dpp<kDppXor1>(o));
    o = max(o, dpp<kDppXor2>(o));
    o = max(o, dpp<kDppRor4>(o));
    return ord2f(max(o, dpp<kDppRor8>(o)));
}
__device__ __forceinline__ int row_sum(int x) {
    x += dpp<kDppXor1>(x);
    x += dpp<kDppXor2>(x);
    x += dpp<kDppRor4>(x);
    return x + dpp<kDppRor8>(x);
}
__device__ __forceinline__ uint32_t row_or(uint32_t x) {
    x |= (uint32_t)dpp<kDppXor1>((int)x);
    x |= (uint32_t)dpp<kDppXor2>((int)x);
    x |= (uint32_t)dpp<kDppRor4>((int)x);
    return x | (uint32_t)dpp<kDppRor8>((int)x);
}
// inclusive prefix sum within the row
__device__ __forceinline__ int row_scan(int x) {
    x += dpp<kDppShr1>(x);
    x += dpp<kDppShr2>(x);
    x += dpp<kDppShr4>(x);
    return x + dpp<kDppShr8>(x);
}

}  // namespace pg
