// Post chain for gfx950: the HIP counterpart of the offscreen passes that consume the cloud image,
// god-ray.frag:41-76 -> radialBlur.frag:36-63 -> tonemap.frag:11-34 (VulkanApplication.cpp:938-966).
//
// Three launches of blocks of 256 work-items (16x16 pixels; 64x16 for the god rays), one contiguous band of
// tiles per XCD:
//   alpha_plane_kernel  the cloud image's alpha as a plane of floats (16 B read, 4 B written);
//   god_ray_kernel      four pixels a work-item: 9 bilinear taps of that plane each (centre + 8 toward
//                       the sun), writes the alpha plane of framebuffer 1 (4 B/pixel);
//   blur_tonemap_kernel one work-item per pixel: bilinear centre tap of the image's RGB, 10 bilinear
//                       taps of that alpha plane toward the sun, the radial-blur colour, then the
//                       Uncharted-2 tonemap + vignette, written as RGBA8 (and optionally the HDR
//                       radial-blur value).
// The taps of neighbouring pixels overlap, so after the first touch they come from L2. The algorithmic
// traffic is 16 B read + 4 B written (alpha plane), 4 B read + 4 B written (god rays) and 16 + 4 B
// read + 4 (or 20) B written (radial blur + tonemap) per pixel. The tap kernels are bound by vector operations
// and by the caches' lanes: waves whose taps are all inside the image take a tap without clamps and with one
// 8-byte load a row, and the tonemap of ordinary numbers takes unscaled divisions and no special cases
// (1080p with the HDR output: god rays 29 us -> 17, blur + tonemap 51 -> 38, the chain 78 -> 56).
// Arithmetic follows the shaders' evaluation order with IEEE division/sqrt and no contraction; the
// sampler and the other choices GLSL leaves open are the scalar restatement's, so the result is the
// same bit for bit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "mm_internal.hpp"
#include "cr_math.hpp"

namespace {

__device__ __forceinline__ float clampf(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }

// LINEAR / CLAMP_TO_EDGE axis: x = u n - 0.5 rounded to 1/2^bits; i = floor(x) saturated to 32 bits (0 for NaN,
// whose weight f is NaN), texels i and i + 1, clamped.
__device__ __forceinline__ void axis(float u, int n, int bits, int& i0, int& i1, float& f) {
    float x = u * (float)n - 0.5f;
    // division by 2^bits is the exact multiplication by 2^-bits (one rounding either way)
    const float s = (float)(1 << bits), inv = __int_as_float((127 - bits) << 23);
    x = floorf(x * s + 0.5f) * inv;
    const float fl = floorf(x);
    f = x - fl;
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(fl));
    i0 = min(max(i, 0), n - 1);
    i1 = min(max(i, -1), n - 2) + 1;
}

// Taps of which every texel exists, weights of 1/256 (about 70 issue cycles against 190 for tap_edge): no clamps,
// one 8-byte load a row. u (256 n) - 128 is 256 times u n - 0.5 with the same roundings, and k = floor(that + 0.5)
// holds the texel (k >> 8) and 256 times its weight (k & 255). The exact floor_half_up is the floor of the sum rounded
// to float, as the restatement takes it, for every v here: at most 2^22 (256 texels of 16384), where 0.5 is a
// multiple of the sum's last place, and, as a difference from 128, a multiple of 2^-17, so no v lies so close
// under 0.5 that the sum would round up to 1 (tests/c/cvt_gpu_check.hip compares the two over all of them).
struct Map {
    float w256, h256;  // in vector registers: a float instruction with a scalar operand issues at half the rate
    float right, bottom;
    uint32_t rowBytes;
    bool use;  // offsets into the image fit 32 bits, rows and bytes a row 24, 256 n is exact
};
__device__ __forceinline__ Map make_map(const mm::PostConsts& c) {
    Map m;
    m.w256 = 256.0f * (float)c.width;
    m.h256 = 256.0f * (float)c.height;
    asm("" : "+v"(m.w256), "+v"(m.h256));
    m.right = 256.0f * (float)(c.width - 1) - 1.0f;
    m.bottom = 256.0f * (float)(c.height - 1) - 1.0f;
    m.rowBytes = (uint32_t)c.pitch * 4u;
    m.use = c.bits == 8 && c.width <= 16384 && c.height <= 16384 && c.pitch < (1 << 20) &&
            (uint64_t)c.pitch * (uint32_t)c.height < (1u << 28);
    return m;
}
struct At {
    float x, y;  // 256 times the texel coordinates
};
__device__ __forceinline__ At locate(const Map& m, float u, float v) { return At{u * m.w256 - 128.0f, v * m.h256 - 128.0f}; }
// k <= 256 (n - 1) - 1, so k >> 8 <= n - 2; false for NaN.
__device__ __forceinline__ bool inside(const Map& m, const At& a) {
    return a.x >= 0.0f && a.y >= 0.0f && a.x <= m.right && a.y <= m.bottom;
}
// RN(n / d) from y = RN(1 / d), as div_rn_normal.
__device__ __forceinline__ float div_by(float n, float d, float y) {
    float q = n * y;
    q = __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}
__device__ __forceinline__ bool all_lanes(bool b) { return __builtin_amdgcn_ballot_w64(!b) == 0; }

__device__ __forceinline__ float lerp_r(float a, float b, float t) { return a + t * (b - a); }

// Bilinear tap of a plane of floats.
__device__ __forceinline__ float tap_edge(const float* __restrict__ img, const mm::PostConsts& c, float u, float v) {
    int x0, x1, y0, y1;
    float fx, fy;
    axis(u, c.width, c.bits, x0, x1, fx);
    axis(v, c.height, c.bits, y0, y1, fy);
    const uint32_t r0 = (uint32_t)y0 * (uint32_t)c.pitch, r1 = (uint32_t)y1 * (uint32_t)c.pitch;
    const float t00 = img[r0 + (uint32_t)x0], t01 = img[r0 + (uint32_t)x1];
    const float t10 = img[r1 + (uint32_t)x0], t11 = img[r1 + (uint32_t)x1];
    return lerp_r(lerp_r(t00, t01, fx), lerp_r(t10, t11, fx), fy);
}
__device__ __forceinline__ void texel(const At& a, int& kx, int& ky, float& fx, float& fy) {
    kx = floor_half_up(a.x);
    ky = floor_half_up(a.y);
    fx = (float)(kx & 255) * (1.0f / 256.0f);
    fy = (float)(ky & 255) * (1.0f / 256.0f);
}
__device__ __forceinline__ float tap_inside(const float* __restrict__ img, const Map& m, const At& a) {
    struct __attribute__((packed, aligned(4))) Pair {
        float l, r;
    };
    int kx, ky;
    float fx, fy;
    texel(a, kx, ky, fx, fy);
    const uint32_t off = __umul24((uint32_t)ky >> 8, m.rowBytes) + (((uint32_t)kx >> 6) & ~3u);
    const Pair p = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(img) + off);
    const Pair q = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(img) + m.rowBytes + off);
    return lerp_r(lerp_r(p.l, p.r, fx), lerp_r(q.l, q.r, fx), fy);
}

// One row of tap_inside: two neighbouring texels `off` bytes into a line.
__device__ __forceinline__ float row_filter(const float* __restrict__ line, uint32_t off, float fx) {
    struct __attribute__((packed, aligned(4))) Pair {
        float l, r;
    };
    const Pair p = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(line) + off);
    return lerp_r(p.l, p.r, fx);
}

// The RGB of one bilinear tap of the RGBA image (one 16-byte load per texel).
__device__ __forceinline__ void lerp_rgb(const float4& t00, const float4& t01, const float4& t10, const float4& t11,
                                         float fx, float fy, float rgb[3]) {
    rgb[0] = lerp_r(lerp_r(t00.x, t01.x, fx), lerp_r(t10.x, t11.x, fx), fy);
    rgb[1] = lerp_r(lerp_r(t00.y, t01.y, fx), lerp_r(t10.y, t11.y, fx), fy);
    rgb[2] = lerp_r(lerp_r(t00.z, t01.z, fx), lerp_r(t10.z, t11.z, fx), fy);
}
__device__ __forceinline__ void tap_rgb(const float4* __restrict__ img, const mm::PostConsts& c, const Map& m, float u,
                                        float v, float rgb[3]) {
    float fx, fy;
    const At a = locate(m, u, v);
    if (m.use && all_lanes(inside(m, a))) {
        int kx, ky;
        texel(a, kx, ky, fx, fy);
        const uint32_t off = __umul24((uint32_t)ky >> 8, m.rowBytes * 4u) + (((uint32_t)kx >> 4) & ~15u);
        const float4* p = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(img) + off);
        const float4* q = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(img + c.pitch) + off);
        lerp_rgb(p[0], p[1], q[0], q[1], fx, fy, rgb);
        return;
    }
    int x0, x1, y0, y1;
    axis(u, c.width, c.bits, x0, x1, fx);
    axis(v, c.height, c.bits, y0, y1, fy);
    const uint32_t r0 = (uint32_t)y0 * (uint32_t)c.pitch, r1 = (uint32_t)y1 * (uint32_t)c.pitch;
    lerp_rgb(img[r0 + (uint32_t)x0], img[r0 + (uint32_t)x1], img[r1 + (uint32_t)x0], img[r1 + (uint32_t)x1], fx, fy, rgb);
}

// Uncharted-2 curve (tonemap.frag:11-14) with the shader's constant products folded in float.
template <bool NORMAL>
__device__ __forceinline__ float div_rn(float n, float d) {
    return NORMAL ? div_rn_normal(n, d) : __fdiv_rn(n, d);
}
// NORMAL: x in [0, 1e9], so the quotient is in [0.06, 1].
template <bool NORMAL>
__device__ __forceinline__ float uc2(float x) {
    const float A = 0.15f, k05 = 0.1f * 0.5f, k004 = 0.2f * 0.02f, k06 = 0.2f * 0.3f, k0067 = 0.02f / 0.3f;
    return div_rn<NORMAL>(x * (A * x + k05) + k004, x * (A * x + 0.5f) + k06) - k0067;
}

// pow(x, y) = exp2(y log2 x), both written out as float operations (the scalar restatement
// evaluates the same operations in the same order). log2: x = m 2^e with m in [sqrt(1/2), sqrt(2)),
// log2 m by the atanh series in s = (m - 1) / (m + 1) to s^9; exp2: t = n + f,
// 2^f = sqrt(2) 2^(f - 1/2) by the exponential series in g = (f - 1/2) ln 2 to g^7, scaled by 2^n
// exactly. exp2 within 3 ulp, log2 within 1e-6 absolute; pow within 1e-6 relative over the
// tonemap's inputs (the float rounding of y log2 x dominates); the result is quantised to 8 bits.
template <bool NORMAL>  // x a positive normal number
__device__ __forceinline__ float log2_series(float x) {
    int e = 0;
    if constexpr (!NORMAL) {
        if (!(x > 0.0f)) return x == 0.0f ? -INFINITY : __int_as_float(0x7fc00000);
        if (x == INFINITY) return INFINITY;
        if (x < 1.17549435e-38f) {  // subnormal: scale into the normal range
            x = x * 16777216.0f;
            e = -24;
        }
    }
    uint32_t b = __float_as_uint(x);
    e += (int)((b >> 23) & 255u) - 127;
    float m = __uint_as_float((b & 0x007fffffu) | 0x3f800000u);
    if (m > 1.41421356f) {
        m = m * 0.5f;
        e = e + 1;
    }
    const float s = div_rn_normal(m - 1.0f, m + 1.0f);  // 0 or at least 2^-24 by at most 2.5
    const float s2 = s * s;
    float p = 0.320598898f;
    p = p * s2 + 0.412198583f;
    p = p * s2 + 0.577078016f;
    p = p * s2 + 0.961796694f;
    p = p * s2 + 2.88539008f;
    return (float)e + s * p;
}

template <bool NORMAL>  // |t| < 126
__device__ __forceinline__ float exp2_series(float t) {
    if constexpr (!NORMAL) {
        if (t != t) return t;
        if (t >= 128.0f) return INFINITY;
        if (t < -150.0f) return 0.0f;
    }
    const float n = floorf(t);
    const float g = ((t - n) - 0.5f) * 0.693147181f;
    float p = 1.98412698e-4f;
    p = p * g + 1.38888889e-3f;
    p = p * g + 8.33333333e-3f;
    p = p * g + 4.16666667e-2f;
    p = p * g + 0.166666667f;
    p = p * g + 0.5f;
    p = p * g + 1.0f;
    p = p * g + 1.0f;
    return __builtin_amdgcn_ldexpf(p * 1.41421356f, (int)n);
}

// Block -> tile. Workgroups are dealt round-robin to the 8 XCDs (block b runs on XCD b mod 8),
// each with its own L2; the taps of a pixel reach far toward the sun, so tiles that share cache
// lines should share an XCD. Block b takes tile (b mod 8) * per + b / 8 of the row-major tile list
// (per = ceil(tiles / 8)): each XCD marches one contiguous band of tile rows. Returns false for the
// padding blocks past the last tile.
__device__ __forceinline__ bool xcd_tile(const mm::PostConsts& c, int widthLog2, int heightLog2, uint32_t magic, int& x,
                                         int& y) {
    const int gx = (c.width + (1 << widthLog2) - 1) >> widthLog2;
    const int tiles = gx * ((c.height + (1 << heightLog2) - 1) >> heightLog2);
    const int per = (tiles + 7) >> 3;
    const int t = (int)(blockIdx.x & 7u) * per + (int)(blockIdx.x >> 3);
    if (t >= tiles) return false;
    const int row = magic ? (int)__umulhi((uint32_t)t, magic) : t / gx;  // scalar multiply
    x = (t - row * gx) << widthLog2;
    y = row << heightLog2;
    return true;
}
__device__ __forceinline__ bool pixel_16x16(const mm::PostConsts& c, int& x, int& y) {
    if (!xcd_tile(c, 4, 4, c.tileMagic, x, y)) return false;
    x += threadIdx.x & 15;
    y += threadIdx.x >> 4;
    return x < c.width && y < c.height;
}

__device__ __forceinline__ uint32_t unorm8(float v) {
    return (uint32_t)(clampf(v, 0.0f, 1.0f) * 255.0f + 0.5f);  // NaN: fmaxf takes 0
}

// The image's alpha as a plane of its own: the god-ray taps then read 4-byte texels (32 per
// 128-byte line instead of 8 RGBA32F ones), which is what keeps their far-reaching taps in cache.
__global__ __launch_bounds__(256) void alpha_plane_kernel(const mm::PostConsts c, const float4* __restrict__ img,
                                                          float* __restrict__ plane) {
    int x, y;
    if (!pixel_16x16(c, x, y)) return;
    const uint32_t i = (uint32_t)y * (uint32_t)c.pitch + (uint32_t)x;
    plane[i] = img[i].w;
}

// A wave takes 64 columns of R rows, R pixels a lane. A tap's x depends on the column alone and its y on the row
// alone: a lane's pixels share the x, and the rows' y are computed by lanes 0 .. R - 1 (lane mod R) and read back
// as scalars. The R footprints of a tap together cover at most R + 1 rows of texels as long as the rows' taps
// are no farther apart than the rows are (any density up to 1): for R = 4 five 8-byte loads and five horizontal
// filters instead of eight. One pixel a lane of a 16x4 wave was bound by the L1's four lanes a cycle: 22 us at
// 1080p for the nine taps, 17 with R = 4. Images under a million pixels leave the chip idle and wait for their
// loads instead: R = 1 and three taps in flight (the chain, us, at R = 1 / R = 4: 640x360 16.2 / 19.3, 960x540
// 23.4 / 25.0, 1280x720 34.0 / 33.4, 1600x900 47.8 / 43.7, 1920x1080 62.9 / 58.0; R = 4 with three taps: 59.8).
template <int N>
struct Count {
    static constexpr int value = N;
};
template <int RL, int BATCH>
__global__ __launch_bounds__(256) void god_ray_kernel(const mm::PostConsts c, const float* __restrict__ a0,
                                                      float* __restrict__ alpha) {
    constexpr int R = 1 << RL;
    int x, y;
    if (!xcd_tile(c, 6, 2 + RL, RL == 2 ? c.wideTileMagic : 0u, x, y)) return;
    const int lane = (int)(threadIdx.x & 63u);
    const int col = x + lane, row = y + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * R;
    if (row >= c.height) return;  // the whole wave: every lane stays to the end for the scalars
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 1.0f;  // sun below the horizon: the pass writes alpha 1 (god-ray.frag:55-57)
    if (!c.below) {
        const Map m = make_map(c);
        const float u = div_by((float)min(col, c.width - 1) + 0.5f, (float)c.width, c.rw);
        const float v = div_by((float)min(row + (lane & (R - 1)), c.height - 1) + 0.5f, (float)c.height, c.rh);
        float cx = u * 2.0f - 1.0f, cy = v * 2.0f - 1.0f;
        const float dx = (cx - c.sunX) * c.k, dy = (cy - c.sunY) * c.k;
        float decay = 1.0f, sw = c.sw, fade = c.decay;
        asm("" : "+v"(decay), "+v"(sw), "+v"(fade));
        // N taps from tap i on (-1: the pixel's own), their loads in flight together. The taps lie in order on a
        // line: if the outer two are inside, all are.
        auto taps = [&](auto count, int i) {
            constexpr int N = decltype(count)::value;
            float tu[N], tv[N], t[N][R];
            At a[N];
#pragma unroll
            for (int k = 0; k < N; k++) {
                tu[k] = u;
                tv[k] = v;
                if (i + k >= 0) {
                    cx = cx - dx;
                    cy = cy - dy;
                    tu[k] = __builtin_fmaf(cx, 0.5f, 0.5f);
                    tv[k] = __builtin_fmaf(cy, 0.5f, 0.5f);
                }
                a[k] = locate(m, tu[k], tv[k]);
            }
            if (m.use && all_lanes(inside(m, a[0]) && (N == 1 || inside(m, a[N - 1])))) {
                int iy[N][R];
                uint32_t off[N];
                float fx[N], fy[N][R];
                bool near = true;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    int kx, ky;
                    float f;
                    texel(a[k], kx, ky, fx[k], f);
                    off[k] = ((uint32_t)kx >> 6) & ~3u;
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        iy[k][r] = __builtin_amdgcn_readlane(ky, r) >> 8;
                        fy[k][r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), r));
                        if (r > 0) near = near && (unsigned)(iy[k][r] - iy[k][r - 1]) <= 1u;
                    }
                }
                if (near) {
                    float h[N][R + 1];
#pragma unroll
                    for (int k = 0; k < N; k++)
#pragma unroll
                        for (int r = 0; r <= R; r++)  // rows past the last footprint are read as the last row, unused
                            h[k][r] = row_filter(a0 + (size_t)(uint32_t)min(iy[k][0] + r, c.height - 1) * (uint32_t)c.pitch,
                                                 off[k], fx[k]);
#pragma unroll
                    for (int k = 0; k < N; k++)
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            if (r > 0 && iy[k][r] != iy[k][r > 0 ? r - 1 : 0]) {
#pragma unroll
                                for (int l = 0; l + r <= R; l++) h[k][l] = h[k][l + 1];
                            }
                            t[k][r] = lerp_r(h[k][0], h[k][1], fy[k][r]);
                        }
                } else {
#pragma unroll
                    for (int k = 0; k < N; k++)
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const float* line = a0 + (size_t)(uint32_t)iy[k][r] * (uint32_t)c.pitch;
                            t[k][r] = lerp_r(row_filter(line, off[k], fx[k]), row_filter(line + c.pitch, off[k], fx[k]),
                                             fy[k][r]);
                        }
                }
            } else {
#pragma unroll
                for (int k = 0; k < N; k++)
#pragma unroll
                    for (int r = 0; r < R; r++)
                        t[k][r] = tap_edge(a0, c, tu[k], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tv[k]), r)));
            }
#pragma unroll
            for (int k = 0; k < N; k++) {
                const float w = sw * decay;
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = i + k < 0 ? t[k][r] * 0.5f : acc[r] + (t[k][r] * 0.5f) * w;
                if (i + k >= 0) decay = decay * fade;
            }
        };
        int i = -1;
        if constexpr (BATCH > 1)
            for (; i + BATCH <= c.samples; i += BATCH) taps(Count<BATCH>{}, i);
        for (; i < c.samples; i++) taps(Count<1>{}, i);
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = acc[r] * c.godExposure;
    }
    if (col >= c.width) return;
#pragma unroll
    for (int r = 0; r < R; r++)
        if (row + r < c.height) alpha[(uint32_t)(row + r) * (uint32_t)c.pitch + (uint32_t)col] = acc[r];
}

__global__ __launch_bounds__(256) void blur_tonemap_kernel(const mm::PostConsts c, const float4* __restrict__ img,
                                                           const float* __restrict__ alpha, float4* __restrict__ hdr,
                                                           uint32_t* __restrict__ rgba8) {
    int x, y;
    if (!pixel_16x16(c, x, y)) return;
    const Map m = make_map(c);
    const float u = div_by((float)x + 0.5f, (float)c.width, c.rw), v = div_by((float)y + 0.5f, (float)c.height, c.rh);
    float rgb[3];
    tap_rgb(img, c, m, u, v, rgb);
    float o[3] = {rgb[0], rgb[1], rgb[2]};
    if (!c.below) {
        const float sx = u * 2.0f - 1.0f, sy = v * 2.0f - 1.0f;
        float lx = c.sunX - sx, ly = c.sunY - sy;
        const float d2 = lx * lx + ly * ly;
        float dist;
        if (all_lanes(fminf(fabsf(lx), fabsf(ly)) >= 0x1p-40f && d2 <= 0x1p80f)) {  // quotients far from subnormal
            const float y = __builtin_amdgcn_rsqf(d2);
            dist = sqrt_from_rsq(d2, y);
            const float r = rcp_refine(dist, y);
            lx = div_by(lx, dist, r);
            ly = div_by(ly, dist, r);
        } else {
            dist = sqrt_rn(d2);
            lx = __fdiv_rn(lx, dist);
            ly = __fdiv_rn(ly, dist);
        }
        // taps -0.08 .. 0.08 along the line to the sun, in order: if the outer two are inside, all are
        float scale = c.blurScale, gain = c.blurGain;
        asm("" : "+v"(scale), "+v"(gain));
        constexpr float kTaps[5] = {0.08f, 0.05f, 0.03f, 0.02f, 0.01f};
        float tu[10], tv[10], t[10];
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const float ox = ((kTaps[i] * lx) * scale) * dist, oy = ((kTaps[i] * ly) * scale) * dist;
            tu[i] = __builtin_fmaf(sx - ox, 0.5f, 0.5f);
            tv[i] = __builtin_fmaf(sy - oy, 0.5f, 0.5f);
            tu[9 - i] = __builtin_fmaf(sx + ox, 0.5f, 0.5f);
            tv[9 - i] = __builtin_fmaf(sy + oy, 0.5f, 0.5f);
        }
        if (m.use && all_lanes(inside(m, locate(m, tu[0], tv[0])) && inside(m, locate(m, tu[9], tv[9])))) {
#pragma unroll
            for (int i = 0; i < 10; i++) t[i] = tap_inside(alpha, m, locate(m, tu[i], tv[i]));
        } else {
#pragma unroll
            for (int i = 0; i < 10; i++) t[i] = tap_edge(alpha, c, tu[i], tv[i]);
        }
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < 10; i++) acc = acc + t[i] * gain;
        acc = __fdiv_rn(acc, 10.0f);
        for (int k = 0; k < 3; k++) o[k] = c.gc[k] * acc + 0.5f * rgb[k];
    }
    const uint32_t i = (uint32_t)y * (uint32_t)c.pitch + (uint32_t)x;
    if (hdr) hdr[i] = make_float4(o[0], o[1], o[2], 1.0f);
    if (rgba8) {
        const float vx = u - 0.5f, vy = v - 0.5f;
        const float vig = vx * vx + vy * vy;
        // framebuffer 2 sampled at the pixel centre returns this pixel's radial-blur value
        float t[3];
        bool ok = true;
        for (int k = 0; k < 3; k++) {
            t[k] = c.exposure * o[k];
            ok = ok && __float_as_uint(t[k]) <= __float_as_uint(1e9f);  // and not negative, not NaN
        }
        if (all_lanes(ok)) {
            for (int k = 0; k < 3; k++) t[k] = uc2<true>(t[k]) * c.whitemap;
        } else {
            for (int k = 0; k < 3; k++) t[k] = uc2<false>(t[k]) * c.whitemap;
        }
        ok = __builtin_amdgcn_classf(t[0], 0x100) && __builtin_amdgcn_classf(t[1], 0x100) &&
             __builtin_amdgcn_classf(t[2], 0x100);  // positive normal numbers
        if (all_lanes(ok)) {
            for (int k = 0; k < 3; k++) t[k] = c.invGamma * log2_series<true>(t[k]);  // pow (tonemap.frag:22)
        } else {
            for (int k = 0; k < 3; k++) t[k] = c.invGamma * log2_series<false>(t[k]);
        }
        ok = fabsf(t[0]) < 126.0f && fabsf(t[1]) < 126.0f && fabsf(t[2]) < 126.0f;
        if (all_lanes(ok)) {
            for (int k = 0; k < 3; k++) t[k] = exp2_series<true>(t[k]);
        } else {
            for (int k = 0; k < 3; k++) t[k] = exp2_series<false>(t[k]);
        }
        uint32_t q = 255u << 24;
        for (int k = 0; k < 3; k++) q |= unorm8(t[k] * (1.0f - vig) + c.vignette[k] * vig) << (8 * k);
        rgba8[i] = q;
    }
}

}  // namespace

namespace mm {

int launch_post(const PostConsts& c, const float* image, float* scratch, float* hdr, uint8_t* rgba8, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    const long tiles = (long)((c.width + 15) / 16) * ((c.height + 15) / 16);
    dim3 grid((unsigned)(8 * ((tiles + 7) / 8))), block(256);  // 1-D: xcd_tile maps blocks to tiles
    // scratch: plane 0 = the image's alpha, plane 1 = framebuffer 1's alpha (the god-ray output)
    float* a0 = scratch;
    float* a1 = scratch + (size_t)c.pitch * c.height;
    if (!c.below) hipLaunchKernelGGL(alpha_plane_kernel, grid, block, 0, s, c, (const float4*)image, a0);
    const bool large = (long)c.width * c.height >= 1 << 20;  // see god_ray_kernel
    const int rows = large ? 16 : 4;
    const long wide = (long)((c.width + 63) / 64) * ((c.height + rows - 1) / rows);
    const dim3 wideGrid((unsigned)(8 * ((wide + 7) / 8)));
    if (large) hipLaunchKernelGGL((god_ray_kernel<2, 1>), wideGrid, block, 0, s, c, (const float*)a0, a1);
    else hipLaunchKernelGGL((god_ray_kernel<0, 3>), wideGrid, block, 0, s, c, (const float*)a0, a1);
    hipLaunchKernelGGL(blur_tonemap_kernel, grid, block, 0, s, c, (const float4*)image, (const float*)a1,
                       (float4*)hdr, (uint32_t*)rgba8);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

}  // namespace mm
