// q8_1 quantizer arithmetic shared by the kernels that stage activations.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// value of another lane of the same quad (DPP quad_perm CTRL)
template <int CTRL>
__device__ __forceinline__ float quad_swap(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// q8_1 quantizer arithmetic in fewer operations, bit-identical to the IEEE forms (checked for
// every input of the ranges below by tests/arith/q8_arith_check.c):
//   amax / 127: product with RN(1/127) and one fma correction of its residual (Markstein), for
//     finite amax >= 2^-118 (a normal quotient); other values take the IEEE division;
//   roundf(v) (half away from zero) as a truncating conversion of v + copysign(0.49999997, v),
//     for |v| <= 2^23 (the quantizer's |v| <= 127.x).
__device__ __forceinline__ float q8_div127(float amax) {
    if (__builtin_expect(!(amax >= 0x1p-118f && amax <= 0x1.fffffep127f), 0)) return amax / 127.0f;
    const float c = 1.0f / 127.0f;
    const float q = amax * c;
    return __builtin_fmaf(__builtin_fmaf(-q, 127.0f, amax), c, q);
}
// roundf(x * id) with the product rounded first (no fma contraction, as the check assumes)
__device__ __forceinline__ int q8_round_mul(float x, float id) {
#pragma clang fp contract(off)
    const float v = x * id;
    return (int)(v + __builtin_copysignf(0.49999997f, v));
}

// Exact u / d for 0 <= u < 2^21 through the rounded reciprocal rd = 1/d (two VALU operations
// instead of a ~20-instruction integer division): (u + 0.5) / d lies at least 0.5/d from an
// integer, and the two roundings move it by at most 3 * 2^-24 * (u + 0.5) / d, less than that.
__device__ __forceinline__ int udiv_small(int u, float rd) { return (int)(((float)u + 0.5f) * rd); }
