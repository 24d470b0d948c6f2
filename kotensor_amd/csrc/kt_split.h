// kt_split.h -- fp32 numbers as three bf16 numbers, for fp32-precision products on the bf16
// matrix units (kt_split.hip, the prefill attention in kt_decoder.hip).
#pragma once

#include "kt_common.h"

namespace kt {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes at any alignment (dword accesses need none in global memory).
template <typename T>
__device__ __forceinline__ T load_any(const void* p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

// The upper halves of two floats in one dword: their bf16 truncations.
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
}
// v minus its bf16 truncation, exact. (One v_dot2_f32_bf16 does the same, but runs on the
// matrix unit: four of them beside a 32x32x16 product took 63 cycles, four multiply-adds 38.)
__device__ __forceinline__ float below_upper(float v) {
    return v - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u);
}

// Eight finite fp32 numbers as three bf16 operands, p = part[0] + part[1] + part[2]. An
// infinity makes a NaN of its lower parts; the callers look for NaN sums.
__device__ __forceinline__ void split3(const float (&p)[8], bf16x8 (&part)[3]) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = p[2 * i], b = p[2 * i + 1];
        h[i] = upper_halves(a, b);
        const float ra = below_upper(a), rb = below_upper(b);
        m[i] = upper_halves(ra, rb);
        l[i] = upper_halves(below_upper(ra), below_upper(rb));
    }
    part[0] = __builtin_bit_cast(bf16x8, h);
    part[1] = __builtin_bit_cast(bf16x8, m);
    part[2] = __builtin_bit_cast(bf16x8, l);
}

// The same with each part the nearest bf16 number to what is left, for products of two split
// numbers, whose smallest part products are not formed: the rests are unbiased and at most
// 2^-8 and 2^-17 of the number (cut off, one-signed and up to 2^-7 and 2^-15), so that
// the three products left out are at most 2^-24 of the product, with an rms of 2^-27 on normal
// inputs (cut off 2^-21 and 2^-24, always toward zero). As many instructions either way. A
// number that rounds up to infinity (above 3.39e38) makes a NaN of its lower parts, too.
__device__ __forceinline__ uint32_t nearest_halves(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
__device__ __forceinline__ void split3_nearest(const float (&p)[8], bf16x8 (&part)[3]) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        auto below = [](float v, uint32_t half) { return v - __builtin_bit_cast(float, half); };
        h[i] = nearest_halves(p[2 * i], p[2 * i + 1]);
        const float ra = below(p[2 * i], h[i] << 16), rb = below(p[2 * i + 1], h[i] & 0xFFFF0000u);
        m[i] = nearest_halves(ra, rb);
        l[i] = nearest_halves(below(ra, m[i] << 16), below(rb, m[i] & 0xFFFF0000u));
    }
    part[0] = __builtin_bit_cast(bf16x8, h);
    part[1] = __builtin_bit_cast(bf16x8, m);
    part[2] = __builtin_bit_cast(bf16x8, l);
}

}  // namespace kt
