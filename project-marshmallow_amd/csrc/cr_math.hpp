// Correctly rounded single-precision square root and reciprocal for gfx950 device code.
//
// v_sqrt_f32 and v_rcp_f32 are accurate to 1 ulp, and the compiler lowers sqrtf / __fsqrt_rn to the
// former (with denormal scaling only). The scalar restatements round every square root and division
// correctly (IEEE 754), and in the Earth-radius geometry a 1-ulp difference in a normalisation moves
// a sample by ~0.5 m, so the kernels use these instead. tests/c/rn_math_check.c checks the square root's
// selection and tests/c/rn_rsq_check.c the forms built on v_rsq_f32 / v_rcp_f32, on the CPU over every
// mantissa from every 1-ulp start; tests/c/rn_gpu_check.hip checks the results on the GPU over every float.
//
// Issue cycles, measured on a full SIMD (6 waves of one instruction each, MI355X): f32 add / mul / fma,
// integer add, and / or / xor and right shifts 2.5; compares, min / max, conversions, integer multiplies,
// left shifts, byte permutes and any instruction with an SGPR operand 4.3; rcp / rsq / sqrt / exp / log 8.3.
#pragma once
#include <hip/hip_runtime.h>

// RN(sqrt(x)) for x = 0 or x >= 2^-96: take the hardware result s and test the residuals x - s' * s of
// its two neighbours s' (exact through FMA) to pick the correctly rounded value.
__device__ __forceinline__ float sqrt_rn_normal(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float down = __int_as_float(__float_as_int(s) - 1);
    const float up = __int_as_float(__float_as_int(s) + 1);
    const float vd = __builtin_fmaf(-down, s, x);
    const float vu = __builtin_fmaf(-up, s, x);
    const float r = vd <= 0.0f ? down : s;
    return vu > 0.0f ? up : r;
}

// RN(sqrt(x)) for any x >= 0: inputs below 2^-96 are scaled by 2^32 first (result by 2^-16) so
// v_sqrt_f32 never sees a denormal.
__device__ __forceinline__ float sqrt_rn(float x) {
    const bool tiny = x < 0x1p-96f;
    const float r = sqrt_rn_normal(tiny ? x * 0x1p32f : x);
    return tiny ? r * 0x1p-16f : r;
}

// RN(1 / s) for |s| in [2^-125, 2^125]: v_rcp_f32 with its last mantissa bit set (still within 2 ulp), e = 1 - s y
// exactly through FMA, then y + e (y + e y), one power of e more than a Newton step. Correctly rounded from
// every start within 1 ulp, with no special case: the plain step y + e y stops one ulp short when the
// mantissa of s is all ones (1 / s lies just above the midpoint of 2^k and its upper neighbour and the step
// from 2^k ties to even), and setting the bit keeps the start off that tie. An "or" and an FMA cost 5 issue
// cycles of a SIMD; testing for that mantissa and selecting the value cost 14.
__device__ __forceinline__ float rcp_refine(float s, float start) {
    const float y = __uint_as_float(__float_as_uint(start) | 1u);
    const float e = __builtin_fmaf(-s, y, 1.0f);
    return __builtin_fmaf(e, __builtin_fmaf(e, y, y), y);
}
__device__ __forceinline__ float rcp_rn(float s) { return rcp_refine(s, __builtin_amdgcn_rcpf(s)); }

// RN(sqrt(x)) from y = v_rsq_f32(x), for x in [2^-96, 2^96]: g = x y, then g + (x - g^2) y / 2 (one Heron
// step, the residual exact through FMA). x = 0 gives NaN (0 * inf): the callers clamp it to 0 or divide by
// it. Four full-rate instructions after the one transcendental (19 issue cycles); the neighbour selection of
// sqrt_rn_normal takes 33, two of them compares whose result the selects must wait for. From a start
// within 1 ulp exactly one (mantissa, start) pair of 33.5 M rounds the other way on the CPU; v_rsq_f32 of
// gfx950 does not give that start: its results are checked over every float of the range.
__device__ __forceinline__ float sqrt_from_rsq(float x, float y) {
    const float g = x * y, h = 0.5f * y;
    const float d = __builtin_fmaf(-g, g, x);
    return __builtin_fmaf(d, h, g);
}
__device__ __forceinline__ float sqrt_rn_rsq(float x) { return sqrt_from_rsq(x, __builtin_amdgcn_rsqf(x)); }

// RN(1 / RN(sqrt(x))), x in [2^-96, 2^96]: both roundings from one v_rsq_f32 (its result is within 2 ulp
// of the reciprocal of the rounded root, which rcp_refine takes). 29 issue cycles against 60 for
// rcp_rn(sqrt_rn_normal(x)) with the compares and selects.
__device__ __forceinline__ float rcp_sqrt_rn(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    return rcp_refine(sqrt_from_rsq(x, y), y);
}

// RN(n / d) for d and the quotient well inside the normal range (no scaling): y = RN(1 / d), two corrected
// quotients. The first is within 1 ulp, so the second residual is exact and the last FMA rounds the exact
// quotient (Markstein's theorem). 32 issue cycles against 42 for the scaled IEEE sequence.
__device__ __forceinline__ float div_rn_normal(float n, float d) {
    const float y = rcp_rn(d);
    float q = n * y;
    q = __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}

// Two values, as FP8 e4m3 (OCP: bias 7, max finite 448, no infinities), in the low or high half of r: negative
// values and NaN give 0, the conversion rounds to nearest even, subnormals included. tests/c/cvt_gpu_check.hip
// compares it with the rounding written out over every float.
template <bool HIGH>
__device__ __forceinline__ unsigned fp8_pair(float a, float b, unsigned r) {
    a = fminf(fmaxf(a, 0.0f), 448.0f);
    b = fminf(fmaxf(b, 0.0f), 448.0f);
    return (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, (int)r, HIGH);
}

// floor(v + 0.5), exactly (the addition is not rounded to float), for |v| below 2^31.
__device__ __forceinline__ int floor_half_up(float v) {
    int k;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(k) : "v"(v));
    return k;
}
