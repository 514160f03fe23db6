/* CPU check of the correctly rounded forms built on v_rsq_f32 and v_rcp_f32 (csrc/cr_math.hpp): for every
 * float mantissa and every start within 1 ulp, rcp_refine must return RN(1 / s) from a reciprocal start,
 * and RN(1 / RN(sqrt(x))) from a reciprocal-square-root start; sqrt_from_rsq must return RN(sqrt(x)) but for
 * the one (mantissa, start) pair named in its comment. div_rn_normal is checked against the IEEE quotient
 * on seeded operands of the march's remap (n in (0, d], d in [2^-24, 1]) and on all-ones divisors. Built
 * with gcc -mfma; prints the counts and exits non-zero on any other miss. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float fb(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t bf(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

static float rcp_refine(float s, float start) {
    float y = fb(bf(start) | 1u);
    float e = fmaf(-s, y, 1.0f);
    return fmaf(e, fmaf(e, y, y), y);
}
static float sqrt_from_rsq(float x, float y) {
    float g = x * y, h = 0.5f * y;
    return fmaf(fmaf(-g, g, x), h, g);
}
static float div_rn_normal(float n, float d, float start) {
    float y = rcp_refine(d, start), q = n * y;
    q = fmaf(fmaf(-d, q, n), y, q);
    return fmaf(fmaf(-d, q, n), y, q);
}

static double ulp_of(double v) { int e; frexp(v, &e); return ldexp(1.0, e - 24); }
static int within_1ulp(double start, double exact) {
    return fabs(start - exact) <= ulp_of(start < exact ? start : exact);
}

int main(void) {
    long n = 0, bad = 0;
    for (uint32_t m = 0; m < (1u << 23); m++) {
        float s = fb(0x3f800000u | m);
        double exact = 1.0 / (double)s;
        float rn = (float)exact;
        for (int d = -3; d <= 3; d++) {
            float y0 = fb(bf(rn) + d);
            if (!within_1ulp((double)y0, exact)) continue;
            n++;
            bad += rcp_refine(s, y0) != rn;
        }
    }
    printf("reciprocal: %ld starts, %ld misses\n", n, bad);
    long n2 = 0, root = 0, inv = 0;
    for (uint32_t m = 0; m < (1u << 24); m++) {
        float x = fb(0x3f800000u + m), s = sqrtf(x);
        double exact = 1.0 / sqrt((double)x);
        float rn = (float)exact, ri = (float)(1.0 / (double)s);
        for (int d = -2; d <= 2; d++) {
            float y0 = fb(bf(rn) + d);
            if (!within_1ulp((double)y0, exact)) continue;
            n2++;
            root += sqrt_from_rsq(x, y0) != s;
            inv += rcp_refine(s, y0) != ri;
        }
    }
    printf("root: %ld starts, %ld misses; its reciprocal: %ld misses\n", n2, root, inv);
    long n3 = 0, quot = 0;
    uint32_t h = 12345u;
    for (long i = 0; i < 20000000; i++) {
        h = h * 1664525u + 1013904223u;
        float a = (float)(h >> 8) * 0x1p-24f;
        if (i % 16 == 0) a = 0x1p-24f * (float)(1 + (i / 16) % 64);          /* 1 - a all ones and its neighbours */
        if (i % 16 == 1) a = 1.0f - 0x1p-24f * (float)(1 + (i / 16) % 64);   /* the smallest divisors */
        h = h * 1664525u + 1013904223u;
        float v = a + (1.0f - a) * ((float)(h >> 8) * 0x1p-24f);
        if (i % 7 == 0) v = ldexpf(1.0f, -(int)(h % 20)) + a;
        if (!(v > a) || v > 1.0f) continue;
        float num = v - a, den = 1.0f - a, rn = (float)(1.0 / (double)den), q = num / den;
        for (int d = -1; d <= 1; d++) {
            float y0 = fb(bf(rn) + d);
            if (!within_1ulp((double)y0, 1.0 / (double)den)) continue;
            n3++;
            quot += div_rn_normal(num, den, y0) != q;
        }
    }
    printf("quotient: %ld starts, %ld misses\n", n3, quot);
    return bad == 0 && root <= 1 && inv == 0 && quot == 0 ? 0 : 1;
}
