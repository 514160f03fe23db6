// Noise-texture generators for gfx950: curl map, low-res Perlin-Worley/Worley volume, hi-res
// Worley volume and weather map, written directly in the march's storage formats and layouts.
//
// Built with -ffp-contract=off and IEEE division/sqrt so every float/double operation rounds as in
// the CPU restatement: outputs are equal byte for byte.
//
// Curl map: restates GenerateCurlNoise (ImageUtils.cpp:176-223). hashNoise (ImageUtils.cpp:25-29)
// only ever sees integer lattice coordinates in [-1, 24] (pt in [-EPS, 1) times freq <= 24), so the
// gradient index of every lattice point is tabulated once per call (27^3 entries) and the 48
// Perlin evaluations per texel read the table. The global per-channel min/max of the curl field
// is reduced with atomics on order-preserving integer encodings, then a second pass quantises.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <float.h>
#include <algorithm>
#include <mutex>
#include "mm_internal.hpp"
#include "cr_math.hpp"

namespace {

// ------------------------------------------------------------------ curl (ImageUtils.cpp)
constexpr int kLat = 27;       // lattice coordinates -1 .. 25
constexpr int kLatOff = 1;

__device__ __forceinline__ double sin_poly(double x) {
    const double invpio2 = 6.36619772367581382433e-01;
    const double pio2_1 = 1.57079632673412561417e+00;
    const double pio2_1t = 6.07710050650619224932e-11;
    double k = rint(x * invpio2);
    double r = (x - k * pio2_1) - k * pio2_1t;
    double r2 = r * r;
    double s = r + r * r2 * (-1.0 / 6.0 + r2 * (1.0 / 120.0 + r2 * (-1.0 / 5040.0 + r2 * (1.0 / 362880.0
               + r2 * (-1.0 / 39916800.0 + r2 * (1.0 / 6227020800.0 + r2 * (-1.0 / 1307674368000.0)))))));
    double c = 1.0 + r2 * (-0.5 + r2 * (1.0 / 24.0 + r2 * (-1.0 / 720.0 + r2 * (1.0 / 40320.0
               + r2 * (-1.0 / 3628800.0 + r2 * (1.0 / 479001600.0 + r2 * (-1.0 / 87178291200.0
               + r2 * (1.0 / 20922789888000.0))))))));
    long q = ((long)k) & 3;
    if (q == 0) return s;
    if (q == 1) return c;
    if (q == 2) return -s;
    return -c;
}

// Also resets the min / max cells of the field kernel that follows (mm: 3 x (min, max), see f2ord).
__global__ __launch_bounds__(256) void curl_table_kernel(uint8_t* __restrict__ table, uint32_t* __restrict__ mm) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < 6) mm[i] = i & 1 ? 0u : 0xffffffffu;
    if (i >= kLat * kLat * kLat) return;
    const float x = (float)(i % kLat - kLatOff), y = (float)((i / kLat) % kLat - kLatOff),
                z = (float)(i / (kLat * kLat) - kLatOff);
    float px = x * 12.9898f, py = y * 78.233f, pz = z * (float)47.387;
    float d = (px + py) + pz;
    float n = (float)sin_poly((double)d) * 43758.5453f;
    n = n - floorf(n);
    table[i] = (uint8_t)(int)floorf(12.f * n);
}

__constant__ float kBasis[12][3] = {
    {(float)0.7071, (float)0.7071, 0.f},  {(float)0.7071, (float)-0.7071, 0.f},
    {(float)-0.7071, (float)0.7071, 0.f}, {(float)-0.7071, (float)-0.7071, 0.f},
    {(float)0.7071, 0.f, (float)0.7071},  {(float)0.7071, 0.f, (float)-0.7071},
    {(float)-0.7071, 0.f, (float)0.7071}, {(float)-0.7071, 0.f, (float)-0.7071},
    {0.f, (float)0.7071, (float)0.7071},  {0.f, (float)0.7071, (float)-0.7071},
    {0.f, (float)-0.7071, (float)0.7071}, {0.f, (float)-0.7071, (float)-0.7071},
};

__device__ __forceinline__ float ref_lerp(float a, float b, float t) {
    return (float)((1.0 - (double)t) * (double)a + (double)(t * b));
}

__device__ __forceinline__ float grad_dot(const uint8_t* __restrict__ tab, float x, float y, float z, float dx, float dy,
                                          float dz) {
    const int i = ((int)x + kLatOff) + kLat * (((int)y + kLatOff) + kLat * ((int)z + kLatOff));
    const float* g = kBasis[tab[i]];
    float a = g[0] * dx, b = g[1] * dy, c = g[2] * dz;
    return (a + b) + c;
}

// perlinNoise (ImageUtils.cpp:41-73)
__device__ float perlin_ref(const uint8_t* __restrict__ tab, float x, float y, float z, float freq) {
    x *= freq; y *= freq; z *= freq;
    float fx = floorf(x), fy = floorf(y), fz = floorf(z);
    float rx = x - fx, ry = y - fy, rz = z - fz;
    float ux = ((rx * rx) * rx) * ((rx * ((rx * 6.0f) - 15.0f)) + 10.0f);
    float uy = ((ry * ry) * ry) * ((ry * ((ry * 6.0f) - 15.0f)) + 10.0f);
    float uz = ((rz * rz) * rz) * ((rz * ((rz * 6.0f) - 15.0f)) + 10.0f);
    float gx = fx + 1.0f, gy = fy + 1.0f, gz = fz + 1.0f;
    float nnn = grad_dot(tab, fx, fy, fz, rx, ry, rz);
    float nnp = grad_dot(tab, fx, fy, gz, rx - 0.f, ry - 0.f, rz - 1.f);
    float npn = grad_dot(tab, fx, gy, fz, rx - 0.f, ry - 1.f, rz - 0.f);
    float npp = grad_dot(tab, fx, gy, gz, rx - 0.f, ry - 1.f, rz - 1.f);
    float pnn = grad_dot(tab, gx, fy, fz, rx - 1.f, ry - 0.f, rz - 0.f);
    float pnp = grad_dot(tab, gx, fy, gz, rx - 1.f, ry - 0.f, rz - 1.f);
    float ppn = grad_dot(tab, gx, gy, fz, rx - 1.f, ry - 1.f, rz - 0.f);
    float ppp = grad_dot(tab, gx, gy, gz, rx - 1.f, ry - 1.f, rz - 1.f);
    float nn = ref_lerp(nnn, pnn, ux), np = ref_lerp(nnp, pnp, ux);
    float pn = ref_lerp(npn, ppn, ux), pp = ref_lerp(npp, ppp, ux);
    float n = ref_lerp(nn, pn, uy), p = ref_lerp(np, pp, uy);
    return ref_lerp(n, p, uz);
}

// FBM (ImageUtils.cpp:75-87)
__device__ float fbm_ref(const uint8_t* __restrict__ tab, float x, float y, float z, float freq, int octaves) {
    float noise = 0.0f, weight = 1.0f, total = 0.0f;
    for (int i = 0; i < octaves; i++) {
        total += weight;
        noise += weight * perlin_ref(tab, x, y, z, freq);
        freq *= 2.0f;
        weight *= 0.4f;
    }
    return noise / total;
}

__device__ __forceinline__ float central(float a, float b) { return (float)((double)(b - a) / (2.0 * 0.0005)); }

// Order-preserving float <-> uint32 encoding for atomic min/max.
__device__ __forceinline__ uint32_t f2ord(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// curlNoiseFBM (ImageUtils.cpp:130-169) + min/max. A chain of dependent FP64 lerps: latency bounds it, not the
// arithmetic. A block takes 64 texels; its four waves share the six partial derivatives (two FBMs, eight Perlin
// evaluations each) and the first combines them. With a work-item per texel 128^2 took 53-60 us (256 waves of 48
// Perlin evaluations each on 1024 SIMDs).
constexpr int kCurlTexels = 64;
struct CurlArgs {
    uint8_t* table;
    uint32_t* mm;
    float* field;
    int dim;
};
__device__ __forceinline__ void curl_field(const CurlArgs& g, int block, float* lds) {
    float(*part)[kCurlTexels] = reinterpret_cast<float(*)[kCurlTexels]>(lds);  // [6]
    const uint8_t* tab = g.table;
    const int dim = g.dim, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = block * kCurlTexels + lane;
    float* field = g.field;
    uint32_t* mm = g.mm;
    const bool in = i < dim * dim;
    for (int d = wave; d < 6; d += 4) {
        if (!in) continue;
        const int row = i / dim, col = i % dim;
        const float px = (float)col / (float)dim, py = (float)row / (float)dim;
        const double eps = 0.0005;
        const float xm = (float)((double)px - eps), xp = (float)((double)px + eps);
        const float ym = (float)((double)py - eps), yp = (float)((double)py + eps);
        // the derivatives' two points: 0 dydx, 1 dxdy, 2 dxdz, 3 dzdx, 4 dzdy, 5 dydz
        float a[3], b[3];
        switch (d) {
            case 0: a[0] = xm; b[0] = xp; a[1] = b[1] = py; a[2] = b[2] = 0.5f; break;
            case 1: a[0] = b[0] = px; a[1] = ym; b[1] = yp; a[2] = b[2] = 0.5f; break;
            case 2: a[0] = b[0] = px; a[1] = b[1] = 0.5f; a[2] = ym; b[2] = yp; break;
            case 3: a[0] = xm; b[0] = xp; a[1] = b[1] = 0.5f; a[2] = b[2] = py; break;
            case 4: a[0] = b[0] = 0.5f; a[1] = ym; b[1] = yp; a[2] = b[2] = px; break;
            default: a[0] = b[0] = 0.5f; a[1] = b[1] = py; a[2] = xm; b[2] = xp; break;
        }
        part[d][lane] = central(fbm_ref(tab, a[0], a[1], a[2], 3.f, 4), fbm_ref(tab, b[0], b[1], b[2], 3.f, 4));
    }
    __syncthreads();
    if (wave != 0) return;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    if (in) {
        const float v[3] = {part[4][lane] - part[5][lane], part[2][lane] - part[3][lane], part[0][lane] - part[1][lane]};
        for (int k = 0; k < 3; k++) {
            field[3 * i + k] = v[k];
            lo[k] = v[k];
            hi[k] = v[k];
        }
    }
    // wave reduction, then one atomic per block and channel
    for (int k = 0; k < 3; k++) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], off));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], off));
        }
    }
    if (lane == 0) {
        for (int k = 0; k < 3; k++) {
            atomicMin(&mm[2 * k], f2ord(lo[k]));
            atomicMax(&mm[2 * k + 1], f2ord(hi[k]));
        }
    }
}

// remap to [0,1] (ImageUtils.cpp:171-174, 200-204) and quantise (:209-212), written in the
// destination format/layout. FP16x4 keeps the remapped value unquantised.
__global__ __launch_bounds__(256) void curl_store_kernel(const float* __restrict__ field, const uint32_t* __restrict__ mm,
                                                         int dim, int apron, int fmt, uint8_t* __restrict__ dst) {
    const int sd = dim + apron;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= sd * sd) return;
    const int x = i % sd, y = i / sd;
    const int src = (y % dim) * dim + (x % dim);
    float m[3];
    for (int k = 0; k < 3; k++) {
        const float lo = ord2f(mm[2 * k]), hi = ord2f(mm[2 * k + 1]);
        m[k] = 0.f + ((field[3 * src + k] - lo) / (hi - lo) * (1.f - 0.f));
    }
    if (fmt == MM_FMT_RGBA8) {
        uint32_t r = (uint32_t)(uint8_t)(int)roundf(m[0] * 255.f);
        uint32_t g = (uint32_t)(uint8_t)(int)roundf(m[1] * 255.f);
        uint32_t b = (uint32_t)(uint8_t)(int)roundf(m[2] * 255.f);
        reinterpret_cast<uint32_t*>(dst)[i] = r | (g << 8) | (b << 16) | (255u << 24);
    } else {  // MM_FMT_FP16X4
        uint2 v;
        v.x = (uint32_t)__half_as_ushort(__float2half_rn(m[0])) | ((uint32_t)__half_as_ushort(__float2half_rn(m[1])) << 16);
        v.y = (uint32_t)__half_as_ushort(__float2half_rn(m[2]));
        reinterpret_cast<uint2*>(dst)[i] = v;
    }
}

// ------------------------------------------------------------------ build-defined generators
// PCG3D hash (Jarzynski & Olano 2020, "Hash Functions for GPU Rendering").
__device__ __forceinline__ void hash3(uint32_t x, uint32_t y, uint32_t z, uint32_t seed, uint32_t& a, uint32_t& b,
                                      uint32_t& c) {
    uint32_t v0 = x + seed, v1 = y ^ (seed * 0x85EBCA6Bu), v2 = z + (seed * 0xC2B2AE35u);
    v0 = v0 * 1664525u + 1013904223u;
    v1 = v1 * 1664525u + 1013904223u;
    v2 = v2 * 1664525u + 1013904223u;
    v0 += v1 * v2; v1 += v2 * v0; v2 += v0 * v1;
    v0 ^= v0 >> 16; v1 ^= v1 >> 16; v2 ^= v2 >> 16;
    v0 += v1 * v2; v1 += v2 * v0; v2 += v0 * v1;
    a = v0; b = v1; c = v2;
}
__device__ __forceinline__ float u01(uint32_t h) { return (float)(h >> 8) * (1.0f / 16777216.0f); }
// i modulo n, n a power of two as every lattice period here is (4 << octaves): one AND, where the remainder by a
// run-time divisor takes about 25 instructions, three times per hash.
__device__ __forceinline__ int wrapi(int i, int n) { return i & (n - 1); }
__device__ __forceinline__ float clamp01(float v) { return v < 0.f ? 0.f : (v > 1.f ? 1.f : v); }
__device__ __forceinline__ float lerp_(float a, float b, float t) { return a + t * (b - a); }
__device__ __forceinline__ uint32_t layer_seed(uint32_t seed, uint32_t layer) {
    return seed * 0x9E3779B9u + layer * 0x632BE5ABu;
}

// Sources of per-cell data for the Worley and Perlin bodies, addressed by unwrapped cell
// coordinates. HashCells hashes the wrapped cell on the spot; LdsCells reads what a block staged
// in LDS (the same hash of the same wrapped cell, computed once per block), so both feed the same
// arithmetic and give the same bits.
struct HashCells {
    int cells;
    uint32_t seed;
    __device__ __forceinline__ void point(int x, int y, int z, float& ux, float& uy, float& uz) const {
        uint32_t h0, h1, h2;
        hash3((uint32_t)wrapi(x, cells), (uint32_t)wrapi(y, cells), (uint32_t)wrapi(z, cells), seed, h0, h1, h2);
        ux = u01(h0);
        uy = u01(h1);
        uz = u01(h2);
    }
};

struct LdsCells {
    const float4* cell;      // (x, y, z, unused) per staged cell: one 16-byte LDS read per lookup
    int bx, by, bz, nx, ny;  // first staged cell and the staged extent in x and y
    __device__ __forceinline__ void point(int x, int y, int z, float& ux, float& uy, float& uz) const {
        const float4 v = cell[((z - bz) * ny + (y - by)) * nx + (x - bx)];
        ux = v.x;
        uy = v.y;
        uz = v.z;
    }
    __device__ __forceinline__ const float4* at(int x, int y, int z) const {
        return cell + (((z - bz) * ny + (y - by)) * nx + (x - bx));
    }
};

// 1 - min(sqrt(d2), 1). Distances below 2^-48 give 1 like that bound's, so the root needs no special case: 30
// issue cycles against 70, once per Worley level.
__device__ __forceinline__ float inverted(float d2) {
    return 1.0f - sqrt_rn_rsq(__builtin_amdgcn_fmed3f(d2, 0x1p-96f, 1.0f));
}

// A lower bound of fl((b - u)^2) over u in [0, 1], with the same roundings (each is monotone): no cell of a row
// whose bounds in y and z sum to `best` or more can lower it, so the row is skipped and the minimum is the same.
__device__ __forceinline__ float near_sq(float b) {
    const float d = __builtin_fmaxf(__builtin_fmaxf(b - 1.0f, -b), 0.0f);
    return d * d;
}

// Inverted F1 cellular noise on a periodic grid of `cells`^3 cells.
template <class Cells>
__device__ __forceinline__ float worley_at(float px, float py, float pz, int cells, const Cells& src) {
    float qx = px * (float)cells, qy = py * (float)cells, qz = pz * (float)cells;
    int ix = (int)floorf(qx), iy = (int)floorf(qy), iz = (int)floorf(qz);
    float best = 1e30f;
#pragma unroll
    for (int oz = -1; oz <= 1; oz++) {
        const float bz = qz - (float)(iz + oz);
#pragma unroll
        for (int oy = -1; oy <= 1; oy++) {
            const float by = qy - (float)(iy + oy);
#pragma unroll
            for (int ox = -1; ox <= 1; ox++) {
                float ux, uy, uz;
                src.point(ix + ox, iy + oy, iz + oz, ux, uy, uz);
                float dx = (qx - (float)(ix + ox)) - ux;
                float dy = by - uy;
                float dz = bz - uz;
                float d2 = ((dx * dx) + (dy * dy)) + (dz * dz);
                best = __builtin_fminf(d2, best);  // = d2 < best ? d2 : best (no NaN: d2 >= 0)
            }
        }
    }
    return inverted(best);
}

// worley_at over staged cells: the same arithmetic, each row of neighbours at constant offsets from its first.
__device__ __forceinline__ float worley_at(float px, float py, float pz, int cells, const LdsCells& src) {
    const float qx = px * (float)cells, qy = py * (float)cells, qz = pz * (float)cells;
    const int ix = (int)floorf(qx), iy = (int)floorf(qy), iz = (int)floorf(qz);
    const float4* home = src.at(ix - 1, iy, iz);
    float bx[3], best = 1e30f;
#pragma unroll
    for (int o = 0; o < 3; o++) bx[o] = qx - (float)(ix + o - 1);
#pragma unroll
    for (int oz = -1; oz <= 1; oz++) {
        const float bz = qz - (float)(iz + oz);
#pragma unroll
        for (int oy = -1; oy <= 1; oy++) {
            const float by = qy - (float)(iy + oy);
            const float4* row = home + (oz * src.ny + oy) * src.nx;
#pragma unroll
            for (int o = 0; o < 3; o++) {
                const float4 u = row[o];
                const float dx = bx[o] - u.x, dy = by - u.y, dz = bz - u.z;
                best = __builtin_fminf(((dx * dx) + (dy * dy)) + (dz * dz), best);
            }
        }
    }
    return inverted(best);
}

__constant__ float kGrad[12][3] = {{1, 1, 0}, {-1, 1, 0}, {1, -1, 0}, {-1, -1, 0}, {1, 0, 1},  {-1, 0, 1},
                                   {1, 0, -1}, {-1, 0, -1}, {0, 1, 1}, {0, -1, 1}, {0, 1, -1}, {0, -1, -1}};

// Gradient of a lattice point of the periodic Perlin grid, from the hash of the wrapped point.
struct HashGrads {
    int period;
    uint32_t seed;
    __device__ __forceinline__ void point(int x, int y, int z, float& gx, float& gy, float& gz) const {
        uint32_t h0, h1, h2;
        hash3((uint32_t)wrapi(x, period), (uint32_t)wrapi(y, period), (uint32_t)wrapi(z, period), seed, h0, h1, h2);
        const float* g = kGrad[h0 % 12u];
        gx = g[0];
        gy = g[1];
        gz = g[2];
    }
};

__device__ __forceinline__ float fade(float t) { return ((t * t) * t) * ((t * ((t * 6.0f) - 15.0f)) + 10.0f); }

template <class Grads>
__device__ __forceinline__ float perlin_at(float px, float py, float pz, int period, const Grads& src) {
    float qx = px * (float)period, qy = py * (float)period, qz = pz * (float)period;
    float fx = floorf(qx), fy = floorf(qy), fz = floorf(qz);
    float rx = qx - fx, ry = qy - fy, rz = qz - fz;
    int ix = (int)fx, iy = (int)fy, iz = (int)fz;
    float n[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        int dx = c & 1, dy = (c >> 1) & 1, dz = c >> 2;
        float g0, g1, g2;
        src.point(ix + dx, iy + dy, iz + dz, g0, g1, g2);
        float ax = rx - (float)dx, ay = ry - (float)dy, az = rz - (float)dz;
        n[c] = ((g0 * ax) + (g1 * ay)) + (g2 * az);
    }
    float ux = fade(rx), uy = fade(ry), uz = fade(rz);
    float x00 = lerp_(n[0], n[1], ux), x10 = lerp_(n[2], n[3], ux);
    float x01 = lerp_(n[4], n[5], ux), x11 = lerp_(n[6], n[7], ux);
    float y0 = lerp_(x00, x10, uy), y1 = lerp_(x01, x11, uy);
    return lerp_(y0, y1, uz);
}

// The value at lattice point (x, y) of a periodic grid.
__device__ __forceinline__ float value_at(int x, int y, int period, uint32_t seed) {
    uint32_t h0, h1, h2;
    hash3((uint32_t)wrapi(x, period), (uint32_t)wrapi(y, period), 0u, seed, h0, h1, h2);
    return u01(h0);
}
// Value noise; at(x, y) gives the lattice points' values.
template <class At>
__device__ __forceinline__ float value2(float px, float py, int period, const At& at) {
    const float qx = px * (float)period, qy = py * (float)period;
    const float fx = floorf(qx), fy = floorf(qy);
    const float tx = qx - fx, ty = qy - fy;
    const int ix = (int)fx, iy = (int)fy;
    const float sx = (tx * tx) * (3.0f - 2.0f * tx), sy = (ty * ty) * (3.0f - 2.0f * ty);
    return lerp_(lerp_(at(ix, iy), at(ix + 1, iy), sx), lerp_(at(ix, iy + 1), at(ix + 1, iy + 1), sx), sy);
}

__device__ __forceinline__ uint32_t q8(float v) {
    v = clamp01(v);
    return (uint32_t)(int)floorf(v * 255.0f + 0.5f);
}

__device__ __forceinline__ uint32_t half_bits(float v) { return (uint32_t)__half_as_ushort(__float2half_rn(v)); }

__device__ __forceinline__ uint32_t fp8x4(float a, float b, float c, float d) {
    return fp8_pair<true>(c, d, fp8_pair<false>(a, b, 0u));
}

struct GenArgs {
    uint8_t* dst;
    int dim, apron, fmt;
    uint32_t seed;
    float coverage;
    float inv_scale[4];
};

// ---- low-res volume: 4 Perlin octaves (periods 4..32) and 4 Worley layers of 3 octaves
// (cells 4..128). "Level" l < 4 is Perlin octave l, l >= 4 is Worley layer (l - 4) / 3, octave
// (l - 4) % 3; both sources below hand out the lattice data of a level.
constexpr int kLowLevels = 16;
__host__ __device__ constexpr int low_level_cells(int l) {
    return l < 4 ? 4 << l : (4 << ((l - 4) / 3)) << ((l - 4) % 3);
}
__device__ __forceinline__ uint32_t low_level_seed(uint32_t seed, int l) {
    return l < 4 ? layer_seed(seed, 1) + (uint32_t)l : layer_seed(seed, 2 + (uint32_t)(l - 4) / 3) + (uint32_t)((l - 4) % 3);
}

// ---- hi-res volume: 3 Worley layers of 3 octaves (cells 4..64); level l is layer l / 3, octave l % 3.
constexpr int kHiLevels = 9;
__host__ __device__ constexpr int hi_level_cells(int l) { return (4 << (l / 3)) << (l % 3); }
__device__ __forceinline__ uint32_t hi_level_seed(uint32_t seed, int l) {
    return layer_seed(seed, 6 + (uint32_t)l / 3) + (uint32_t)l % 3;
}

// Bricks of the volume kernels (texels per axis, 256 work-items each) and the lattice cells a block may stage
// in LDS at a time (53 KB: three blocks a CU).
constexpr int kBrickX = 8, kBrickY = 8, kBrickZ = 4;
constexpr int kStageCap = 3376;
// A level is staged when its box has fewer cells than the brick's texels would hash between them.
constexpr int kStageLevelCap = 27 * kBrickX * kBrickY * kBrickZ / 2;

// Lattice cells of one level around a brick: cells [b, b + n) per axis, staged at offset `off` (-1: not staged).
struct StageMeta {
    int bx, by, bz, nx, ny, nz, off;
};

// The low-res texel's 32-bit word (RGBA8 or FP8 x 4).
__device__ __forceinline__ uint32_t encode_low_res(const GenArgs& a, const float v[4]) {
    if (a.fmt == MM_FMT_RGBA8) return q8(v[0]) | (q8(v[1]) << 8) | (q8(v[2]) << 16) | (q8(v[3]) << 24);
    return fp8x4(v[0] * a.inv_scale[0], v[1] * a.inv_scale[1], v[2] * a.inv_scale[2], v[3] * a.inv_scale[3]);  // MM_FMT_FP8X4
}

__device__ __forceinline__ void store_hi_res(const GenArgs& a, long i, const float v[3]) {
    if (a.fmt == MM_FMT_RGBA8) {
        reinterpret_cast<uint32_t*>(a.dst)[i] = q8(v[0]) | (q8(v[1]) << 8) | (q8(v[2]) << 16);
    } else {  // MM_FMT_FP16X4
        uint2 o;
        o.x = half_bits(v[0]) | (half_bits(v[1]) << 16);
        o.y = half_bits(v[2]);
        reinterpret_cast<uint2*>(a.dst)[i] = o;
    }
}

__device__ __forceinline__ float worley_mix(float a, float b, float c) { return (0.625f * a + 0.25f * b) + 0.125f * c; }
// A Worley channel of the textures, and the low-res Perlin-Worley one.
__device__ __forceinline__ float worley_channel(float wf) { return clamp01(0.26f + 0.9f * wf); }
__device__ __forceinline__ float perlin_worley_channel(float perlin, float wf) {
    const float p01 = clamp01(0.5f + 1.5f * perlin);
    const float pw = (p01 - (wf - 1.0f)) / (1.0f - (wf - 1.0f));
    return clamp01(0.8f * pw - 0.04f);
}

// Cells [floor(q(t0)) - pad, floor(q(t1)) + 1] of one axis, q(t) = ((2t + 1) / (2 dim)) * cells,
// evaluated as the texel evaluates it (q is monotone in t, so every texel's cells lie inside).
__device__ __forceinline__ void axis_span(int t0, int t1, float inv, int cells, int pad, int& base, int& n) {
    const float q0 = ((float)(2 * t0 + 1) * inv) * (float)cells;
    const float q1 = ((float)(2 * t1 + 1) * inv) * (float)cells;
    base = (int)floorf(q0) - pad;
    n = ((int)floorf(q1) + 1) - base + 1;
}

// Cells of a level's box around a brick of `b` texels per axis, at most (for the host's LDS size).
inline long box_bound(int b, int dim, int cells, int pad) { return ((long)(b - 1) * cells + dim - 1) / dim + 3 + pad; }

// Volumes of any size: a block of 256 work-items takes an 8 x 8 x 4 brick of logical texels, one each. The
// lattice cells the brick's texels touch are hashed once into LDS, layer by layer (the Perlin octaves, then
// each Worley layer's three), while a layer's levels fit `cap` cells and are fewer than half of what the texels
// would hash; the others (small volumes at high frequencies, where cells outnumber texels) hash in place.
// Staging layer by layer, not all levels at once, lets three to eight blocks share a CU: 72^3 low-res 120 us ->
// 85, 32^3 hi-res 20 -> 15. Vector operations bound it (27 distances, 9 operations each, at each Worley level).
// Texels whose coordinate is below the apron width are also written to the apron copy (x + dim, ...).
template <bool HI>
__device__ __forceinline__ void volume_brick(const GenArgs& a, int block, int cap, float4* cells, StageMeta* meta) {
    constexpr int kFirstWorley = HI ? 0 : 4;
    const int tid = threadIdx.x;
    const int nbx = (a.dim + kBrickX - 1) / kBrickX, nby = (a.dim + kBrickY - 1) / kBrickY;
    const int x0 = (block % nbx) * kBrickX, y0 = ((block / nbx) % nby) * kBrickY, z0 = block / (nbx * nby) * kBrickZ;
    const int x1 = min(x0 + kBrickX, a.dim) - 1, y1 = min(y0 + kBrickY, a.dim) - 1, z1 = min(z0 + kBrickZ, a.dim) - 1;
    const float inv = 1.0f / (float)(2 * a.dim);
    auto level_cells = [](int l) { return HI ? hi_level_cells(l) : low_level_cells(l); };
    auto level_seed = [&](int l) { return HI ? hi_level_seed(a.seed, l) : low_level_seed(a.seed, l); };
    // Stages levels l0 .. l0 + n - 1 (every work-item takes part).
    auto stage = [&](int l0, int n) {
        __syncthreads();  // the last layer's cells are no longer read
        if (tid < n) {
            const int l = l0 + tid, c = level_cells(l), pad = l < kFirstWorley ? 0 : 1;
            StageMeta m;
            axis_span(x0, x1, inv, c, pad, m.bx, m.nx);
            axis_span(y0, y1, inv, c, pad, m.by, m.ny);
            axis_span(z0, z1, inv, c, pad, m.bz, m.nz);
            m.off = 0;
            meta[tid] = m;
        }
        __syncthreads();
        int off = 0;
        for (int k = 0; k < n; k++) {
            const StageMeta m = meta[k];
            const int cnt = m.nx * m.ny * m.nz, l = l0 + k, c = level_cells(l);
            const bool fits = cnt <= kStageLevelCap && off + cnt <= cap;  // uniform across the block
            if (tid == 0) meta[k].off = fits ? off : -1;
            if (!fits) continue;
            const uint32_t seed = level_seed(l);
            // e / n by a reciprocal: e + 1/2 is at least 1 / (2 n) from a multiple, far beyond its rounding
            const float rx = 1.0f / (float)m.nx, ry = 1.0f / (float)m.ny;
            for (int e = (tid + 64 * k) & 255; e < cnt; e += 256) {
                const int yz = (int)(((float)e + 0.5f) * rx), jx = e - yz * m.nx;
                const int jz = (int)(((float)yz + 0.5f) * ry), jy = yz - jz * m.ny;
                float u0, u1, u2;
                if (l < kFirstWorley) HashGrads{c, seed}.point(m.bx + jx, m.by + jy, m.bz + jz, u0, u1, u2);
                else HashCells{c, seed}.point(m.bx + jx, m.by + jy, m.bz + jz, u0, u1, u2);
                cells[off + e] = make_float4(u0, u1, u2, 0.0f);
            }
            off += cnt;
        }
        __syncthreads();
    };
    const int x = x0 + (tid & (kBrickX - 1)), y = y0 + ((tid / kBrickX) & (kBrickY - 1)), z = z0 + tid / (kBrickX * kBrickY);
    const bool in = x <= x1 && y <= y1 && z <= z1;
    const float px = (float)(2 * x + 1) * inv, py = (float)(2 * y + 1) * inv, pz = (float)(2 * z + 1) * inv;
    auto lds = [&](int k) {
        const StageMeta& m = meta[k];
        return LdsCells{cells + m.off, m.bx, m.by, m.bz, m.nx, m.ny};
    };
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float perlin = 0.0f;
    if constexpr (!HI) {
        stage(0, 4);
        if (in) {
            float w = 1.0f;
#pragma unroll 1
            for (int l = 0; l < 4; l++) {
                const int c = level_cells(l);
                perlin = perlin + w * (meta[l].off >= 0 ? perlin_at(px, py, pz, c, lds(l))
                                                        : perlin_at(px, py, pz, c, HashGrads{c, level_seed(l)}));
                w = w * 0.5f;
            }
        }
        perlin = perlin * (1.0f / 1.875f);
    }
#pragma unroll 1
    for (int ly = 0; ly < (HI ? 3 : 4); ly++) {
        const int l0 = kFirstWorley + 3 * ly;
        stage(l0, 3);
        if (!in) continue;
        float f[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int o = 0; o < 3; o++) {
            const int c = level_cells(l0 + o);
            const float w = meta[o].off >= 0 ? worley_at(px, py, pz, c, lds(o))
                                             : worley_at(px, py, pz, c, HashCells{c, level_seed(l0 + o)});
            f[0] = o == 0 ? w : f[0];
            f[1] = o == 1 ? w : f[1];
            f[2] = o == 2 ? w : f[2];
        }
        const float wf = worley_mix(f[0], f[1], f[2]);
        const float ch = !HI && ly == 0 ? perlin_worley_channel(perlin, wf) : worley_channel(wf);
        v[0] = ly == 0 ? ch : v[0];
        v[1] = ly == 1 ? ch : v[1];
        v[2] = ly == 2 ? ch : v[2];
        v[3] = ly == 3 ? ch : v[3];
    }
    if (!in) return;
    const uint32_t word = HI ? 0u : encode_low_res(a, v);
    const long sd = a.dim + a.apron;
    for (int cz = 0; cz < 2; cz++) {
        const int zs = z + cz * a.dim;
        if (cz && zs >= sd) break;
        for (int cy = 0; cy < 2; cy++) {
            const int ys = y + cy * a.dim;
            if (cy && ys >= sd) break;
            for (int cx = 0; cx < 2; cx++) {
                const int xs = x + cx * a.dim;
                if (cx && xs >= sd) break;
                const long i = ((long)zs * sd + ys) * sd + xs;
                if constexpr (HI) store_hi_res(a, i, v);
                else reinterpret_cast<uint32_t*>(a.dst)[i] = word;
            }
        }
    }
}

// ---- the 128^3 low-res volume (the configured size). Bricks of 16 x 8 x 8 texels start at multiples of their
// size, and texel t sits at q = (2t + 1) c / 256 in cell units (exact), so a brick of B texels spans
// floor(q1) - floor(q0) = max(B c / 128 - 1, 0) cells at every position: compile-time boxes.
//
// Each work-item takes four consecutive texels along x. They share their home cell at 9 of the 12 Worley levels
// (cells of 4 texels or more), two by two at 64 cells an axis and step one cell each at 128, so every cell's
// position is read from LDS once for the four, and its y and z differences are squared once: per texel and cell
// 5 operations instead of 9 and a quarter to a half of a read. One texel per work-item was bound by its
// 356 16-byte LDS reads: 250 us a volume, now 114-127, of which about 70 are the distances' vector operations.
// 36 KB of LDS and at most 128 registers, so that four blocks share a CU: 2 x 1024 blocks fill the chip twice
// (three a CU, all levels staged at once: 128-140 us, and the small grids of the other maps waited for slots).
constexpr int k128X = 16, k128Y = 8, k128Z = 8, k128T = 4;
constexpr int k128Span(int l, int b) { return b * low_level_cells(l) / 128 >= 1 ? b * low_level_cells(l) / 128 - 1 : 0; }
constexpr int k128N(int l, int b) { return k128Span(l, b) + 2 + (l < 4 ? 0 : 1); }
constexpr int k128Cells(int l) { return k128N(l, k128X) * k128N(l, k128Y) * k128N(l, k128Z); }
// Levels are staged layer by layer (Perlin 0..3, then three Worley levels at a time) into the same cells.
constexpr bool k128First(int l) { return l == 0 || (l >= 4 && (l - 4) % 3 == 0); }
constexpr int k128Off(int l) { return k128First(l) ? 0 : k128Off(l - 1) + k128Cells(l - 1); }
constexpr int k128LdsCells() {
    int n = 0;
    for (int l = 0; l < kLowLevels; l++) n = k128Off(l) + k128Cells(l) > n ? k128Off(l) + k128Cells(l) : n;
    return n;
}
static_assert(k128N(15, 16) == 18 && k128N(15, 8) == 10 && k128N(0, 8) == 2, "128^3 staged box sizes");
static_assert(k128X / k128T * k128Y * k128Z == 256, "four texels per work-item");
// Home cell of texel t of a work-item's four, relative to the first's.
constexpr int k128Shift(int l, int t) { return low_level_cells(l) == 128 ? t : low_level_cells(l) == 64 ? t / 2 : 0; }

// First cell of level l's box on an axis: floor(q(t0)) - pad for a brick starting at texel t0.
template <int L>
__device__ __forceinline__ int origin128(int t0) { return ((t0 * low_level_cells(L)) >> 7) - (L < 4 ? 0 : 1); }

template <int L>
__device__ __forceinline__ void stage128(float4* cells, uint32_t seed, int x0, int y0, int z0) {
    constexpr int c = low_level_cells(L), nx = k128N(L, k128X), ny = k128N(L, k128Y), off = k128Off(L), n = k128Cells(L);
    const uint32_t s = low_level_seed(seed, L);
    const int bx = origin128<L>(x0), by = origin128<L>(y0), bz = origin128<L>(z0);
    for (int e = ((int)threadIdx.x + 64 * L) & 255; e < n; e += 256) {
        const int jx = e % nx, jy = (e / nx) % ny, jz = e / (nx * ny);
        float u0, u1, u2;
        if constexpr (L < 4) HashGrads{c, s}.point(bx + jx, by + jy, bz + jz, u0, u1, u2);
        else HashCells{c, s}.point(bx + jx, by + jy, bz + jz, u0, u1, u2);
        cells[off + e] = make_float4(u0, u1, u2, 0.0f);
    }
    if constexpr (L + 1 < kLowLevels && !k128First(L + 1)) stage128<L + 1>(cells, seed, x0, y0, z0);
}

// worley_at for the four texels: the same arithmetic for each.
template <int L>
__device__ __forceinline__ void worley128(const float4* cells, const float (&px)[k128T], float py, float pz, int x0,
                                          int y0, int z0, float (&out)[k128T]) {
    constexpr int c = low_level_cells(L), nx = k128N(L, k128X), ny = k128N(L, k128Y), off = k128Off(L);
    const float qy = py * (float)c, qz = pz * (float)c;
    const int iy = (int)floorf(qy), iz = (int)floorf(qz), ix = (int)floorf(px[0] * (float)c);
    const float4* home = cells + off + ((iz - origin128<L>(z0)) * ny + (iy - origin128<L>(y0))) * nx + (ix - origin128<L>(x0));
    float bx[k128T][3], best[k128T];
#pragma unroll
    for (int t = 0; t < k128T; t++) {
        best[t] = 1e30f;
#pragma unroll
        for (int o = 0; o < 3; o++) bx[t][o] = px[t] * (float)c - (float)(ix + k128Shift(L, t) + o - 1);
    }
    float by[3], ly[3];
#pragma unroll
    for (int o = 0; o < 3; o++) {
        by[o] = qy - (float)(iy + o - 1);
        ly[o] = near_sq(by[o]);
    }
    float far = 1e30f;
    // a loop: twelve levels unrolled in full would not fit the instruction cache
#pragma unroll 1
    for (int k = 0; k < 3; k++) {  // slabs 0, -1, +1
        const int oz = k == 0 ? 0 : 2 * k - 3;
        const float bz = qz - (float)(iz + oz), lz = near_sq(bz);
#pragma unroll
        for (int r = 0; r < 3; r++) {  // rows 0, -1, +1
            const int o1 = r == 0 ? 1 : 2 * r - 2;
            if (!(ly[o1] + lz < far)) continue;
#pragma unroll
            for (int j = 0; j < 3 + k128Shift(L, k128T - 1); j++) {
                const float4 u = home[(oz * ny + o1 - 1) * nx + j - 1];
                const float dy = by[o1] - u.y, dz = bz - u.z;
                const float dy2 = dy * dy, dz2 = dz * dz;
#pragma unroll
                for (int t = 0; t < k128T; t++) {
                    const int o = j - k128Shift(L, t);
                    if (o < 0 || o > 2) continue;
                    const float dx = bx[t][o] - u.x;
                    best[t] = __builtin_fminf(((dx * dx) + dy2) + dz2, best[t]);
                }
            }
            far = __builtin_fmaxf(__builtin_fmaxf(best[0], best[1]), __builtin_fmaxf(best[2], best[3]));
        }
    }
#pragma unroll
    for (int t = 0; t < k128T; t++) {
        out[t] = inverted(best[t]);
    }
    __builtin_amdgcn_sched_barrier(0);  // one level's reads in flight at a time: the levels together would spill
}

// perlin_at for the four texels, which share their lattice cell at every Perlin level.
template <int L>
__device__ __forceinline__ void perlin128(const float4* cells, const float (&px)[k128T], float py, float pz, int x0,
                                          int y0, int z0, float (&out)[k128T]) {
    constexpr int c = low_level_cells(L), nx = k128N(L, k128X), ny = k128N(L, k128Y), off = k128Off(L);
    const float qy = py * (float)c, qz = pz * (float)c;
    const float fx = floorf(px[0] * (float)c), fy = floorf(qy), fz = floorf(qz);
    const float ry = qy - fy, rz = qz - fz, uy = fade(ry), uz = fade(rz);
    const float4* home = cells + off + (((int)fz - origin128<L>(z0)) * ny + ((int)fy - origin128<L>(y0))) * nx +
                         ((int)fx - origin128<L>(x0));
    float4 g[8];
#pragma unroll
    for (int k = 0; k < 8; k++) g[k] = home[((k >> 2) * ny + ((k >> 1) & 1)) * nx + (k & 1)];
#pragma unroll
    for (int t = 0; t < k128T; t++) {
        const float rx = px[t] * (float)c - fx, ux = fade(rx);
        float n[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float ax = rx - (float)(k & 1), ay = ry - (float)((k >> 1) & 1), az = rz - (float)(k >> 2);
            n[k] = ((g[k].x * ax) + (g[k].y * ay)) + (g[k].z * az);
        }
        const float x00 = lerp_(n[0], n[1], ux), x10 = lerp_(n[2], n[3], ux);
        const float x01 = lerp_(n[4], n[5], ux), x11 = lerp_(n[6], n[7], ux);
        out[t] = lerp_(lerp_(x00, x10, uy), lerp_(x01, x11, uy), uz);
    }
}

template <int LY>
__device__ __forceinline__ void layer128(float4* cells, uint32_t seed, const float (&px)[k128T], float py, float pz, int x0,
                                         int y0, int z0, const float (&perlin)[k128T], float (&v)[k128T][4]) {
    float a[k128T], b[k128T], c[k128T];
    __syncthreads();  // the last layer's cells are no longer read
    stage128<4 + 3 * LY>(cells, seed, x0, y0, z0);
    __syncthreads();
    worley128<4 + 3 * LY>(cells, px, py, pz, x0, y0, z0, a);
    worley128<5 + 3 * LY>(cells, px, py, pz, x0, y0, z0, b);
    worley128<6 + 3 * LY>(cells, px, py, pz, x0, y0, z0, c);
#pragma unroll
    for (int t = 0; t < k128T; t++) {
        const float wf = worley_mix(a[t], b[t], c[t]);
        v[t][LY] = LY == 0 ? perlin_worley_channel(perlin[t], wf) : worley_channel(wf);
    }
    if constexpr (LY < 3) layer128<LY + 1>(cells, seed, px, py, pz, x0, y0, z0, perlin, v);
}

template <int L>
__device__ __forceinline__ void perlin_fbm128(const float4* cells, const float (&px)[k128T], float py, float pz, int x0,
                                              int y0, int z0, float w, float (&s)[k128T]) {
    float p[k128T];
    perlin128<L>(cells, px, py, pz, x0, y0, z0, p);
#pragma unroll
    for (int t = 0; t < k128T; t++) s[t] = s[t] + w * p[t];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (L < 3) perlin_fbm128<L + 1>(cells, px, py, pz, x0, y0, z0, w * 0.5f, s);
}

__device__ __forceinline__ void low_res_128(const GenArgs& a, int b, float4* cells) {
    constexpr int dim = 128, nbx = dim / k128X, nby = dim / k128Y;
    const int tid = (int)threadIdx.x;
    const int x0 = (b % nbx) * k128X, y0 = (b / nbx % nby) * k128Y, z0 = b / (nbx * nby) * k128Z;
    stage128<0>(cells, a.seed, x0, y0, z0);
    __syncthreads();
    const int x = x0 + (tid % (k128X / k128T)) * k128T, y = y0 + tid / (k128X / k128T) % k128Y,
              z = z0 + tid / (k128X / k128T * k128Y);
    constexpr float inv = 1.0f / (2 * dim);
    float px[k128T];
#pragma unroll
    for (int t = 0; t < k128T; t++) px[t] = (float)(2 * (x + t) + 1) * inv;
    const float py = (float)(2 * y + 1) * inv, pz = (float)(2 * z + 1) * inv;
    float perlin[k128T] = {}, v[k128T][4];
    perlin_fbm128<0>(cells, px, py, pz, x0, y0, z0, 1.0f, perlin);
#pragma unroll
    for (int t = 0; t < k128T; t++) {
        perlin[t] = perlin[t] * (1.0f / 1.875f);
        asm volatile("" : "+v"(perlin[t]));  // computed here: sunk to its use, it would hold 96 registers of gradients
    }
    layer128<0>(cells, a.seed, px, py, pz, x0, y0, z0, perlin, v);
    uint32_t word[k128T];
#pragma unroll
    for (int t = 0; t < k128T; t++) word[t] = encode_low_res(a, v[t]);
    const long sd = dim + a.apron;
    for (int zs = z; zs < sd; zs += dim)
        for (int ys = y; ys < sd; ys += dim) {
            uint32_t* row = reinterpret_cast<uint32_t*>(a.dst) + ((long)zs * sd + ys) * sd + x;
#pragma unroll
            for (int t = 0; t < k128T; t++) row[t] = word[t];
            if (x + dim < sd) row[dim] = word[0];  // the apron repeats texel 0 (x is a multiple of 4)
        }
}

// A block takes 16 x 16 logical texels. The lattice values they touch are hashed once into LDS, level by level
// (three FBMs of five octaves), while they fit; the others hash in place (small maps at high frequencies). 60
// hashes a texel of the 512^2 map were 14.6 us of vector operations, now 10.3 alone.
constexpr int kWeatherTile = 16, kWeatherLevels = 15, kWeatherCap = 4096;
__device__ __forceinline__ int weather_period(int l) { return (l < 5 ? 4 : 8) << (l % 5); }
__device__ __forceinline__ uint32_t weather_seed(uint32_t seed, int l) {
    return layer_seed(seed, 11 + (uint32_t)l / 5) + (uint32_t)l % 5;
}
__device__ __forceinline__ void weather_tile(const GenArgs& a, int block, float* values, StageMeta* meta) {
    const int tid = threadIdx.x, tiles = (a.dim + kWeatherTile - 1) / kWeatherTile;
    const int x0 = block % tiles * kWeatherTile, y0 = block / tiles * kWeatherTile;
    const int x1 = min(x0 + kWeatherTile, a.dim) - 1, y1 = min(y0 + kWeatherTile, a.dim) - 1;
    const float inv = 1.0f / (float)(2 * a.dim);
    if (tid < kWeatherLevels) {
        StageMeta m{};
        axis_span(x0, x1, inv, weather_period(tid), 0, m.bx, m.nx);
        axis_span(y0, y1, inv, weather_period(tid), 0, m.by, m.ny);
        meta[tid] = m;
    }
    __syncthreads();
    int off = 0;
    for (int l = 0; l < kWeatherLevels; l++) {
        const StageMeta m = meta[l];
        const int cnt = m.nx * m.ny;
        const bool fits = cnt <= 2 * kWeatherTile * kWeatherTile && off + cnt <= kWeatherCap;  // uniform across the block
        if (tid == 0) meta[l].off = fits ? off : -1;
        if (!fits) continue;
        if (l % 4 == tid / 64) {  // a wave per level, four at a time
            const float rx = 1.0f / (float)m.nx;  // e / nx as in volume_brick
            for (int e = tid & 63; e < cnt; e += 64) {
                const int jy = (int)(((float)e + 0.5f) * rx);
                values[off + e] = value_at(m.bx + (e - jy * m.nx), m.by + jy, weather_period(l), weather_seed(a.seed, l));
            }
        }
        off += cnt;
    }
    __syncthreads();
    const int x = x0 + tid % kWeatherTile, y = y0 + tid / kWeatherTile;
    if (x > x1 || y > y1) return;
    const float px = (float)(2 * x + 1) * inv, py = (float)(2 * y + 1) * inv;
    float f[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float s = 0.f, w = 1.f;
#pragma unroll 1
        for (int l = 5 * k; l < 5 * k + 5; l++) {
            const int period = weather_period(l);
            const StageMeta m = meta[l];
            const float v = m.off >= 0
                ? value2(px, py, period, [&](int ix, int iy) { return values[m.off + (iy - m.by) * m.nx + (ix - m.bx)]; })
                : value2(px, py, period, [&](int ix, int iy) { return value_at(ix, iy, period, weather_seed(a.seed, l)); });
            s = s + w * v;
            w = w * 0.5f;
        }
        f[k] = s * (1.0f / 1.9375f);
    }
    const float va = f[0], vb = f[1], vc = f[2];
    float r = 0.5f + 2.0f * (va - 0.5f);
    float R = clamp01(r + (a.coverage - 0.5f));
    float G = clamp01(0.5f + 1.5f * ((0.5f * va + 0.5f * vc) - 0.5f));
    float B = clamp01(0.5f + 2.5f * (vb - 0.5f));
    const int sd = a.dim + a.apron;
    for (int ys = y; ys < sd; ys += a.dim)
        for (int xs = x; xs < sd; xs += a.dim) {
            const long i = (long)ys * sd + xs;
            if (a.fmt == MM_FMT_RGBA8) {
                reinterpret_cast<uint32_t*>(a.dst)[i] = q8(R) | (q8(G) << 8) | (q8(B) << 16) | (255u << 24);
            } else {  // MM_FMT_RG8: (coverage, type)
                reinterpret_cast<uint16_t*>(a.dst)[i] = (uint16_t)(q8(R) | (q8(B) << 8));
            }
        }
}

// Every generator in one launch (the curl map's table before it, its store after it): the curl field's blocks, the
// hi-res volume's, the weather map's, then the low-res volume's; any of them may be absent. The small maps'
// latency hides behind the volume. On a stream beside the volume's they waited for slots among its blocks, and
// the fork and the join cost 5 and 16 us: all four maps at 128^3 159 us, in one launch 143.
struct Grids {
    CurlArgs curl;
    GenArgs hi, weather, low;
    int curlBlocks, hiBlocks, weatherBlocks;  // the low-res volume takes the rest
    int hiCap, lowCap;
};
template <bool LOW128>
__global__ __launch_bounds__(256, LOW128 ? 4 : 1) void maps_kernel(Grids g) {
    extern __shared__ float4 cells[];
    __shared__ StageMeta meta[kWeatherLevels];
    int b = (int)blockIdx.x;
    if (b < g.curlBlocks) return curl_field(g.curl, b, reinterpret_cast<float*>(cells));
    b -= g.curlBlocks;
    if (b < g.hiBlocks) return volume_brick<true>(g.hi, b, g.hiCap, cells, meta);
    b -= g.hiBlocks;
    if (b < g.weatherBlocks) return weather_tile(g.weather, b, reinterpret_cast<float*>(cells), meta);
    b -= g.weatherBlocks;
    if constexpr (LOW128) low_res_128(g.low, b, cells);
    else volume_brick<false>(g.low, b, g.lowCap, cells, meta);
}

// ------------------------------------------------------------------ repacking of RGBA8 linear textures
struct PackArgs {
    const uint8_t* src;
    uint8_t* dst;
    int w, h, d;        // logical dims (d = 1 for 2D)
    int apron, fmt, kind;
    float inv_scale[4];
};

__global__ __launch_bounds__(256) void pack_kernel(PackArgs a) {
    const int sw = a.w + a.apron, sh = a.h + a.apron, sdp = (a.d > 1) ? a.d + a.apron : 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)sw * sh * sdp) return;
    const int x = (int)(i % sw) % a.w, y = (int)((i / sw) % sh) % a.h, z = (int)(i / ((long)sw * sh)) % a.d;
    const uint32_t t = reinterpret_cast<const uint32_t*>(a.src)[((long)z * a.h + y) * a.w + x];
    const uint32_t c0 = t & 0xff, c1 = (t >> 8) & 0xff, c2 = (t >> 16) & 0xff, c3 = t >> 24;
    switch (a.fmt) {
        case MM_FMT_RGBA8: reinterpret_cast<uint32_t*>(a.dst)[i] = t; break;
        case MM_FMT_RG8: reinterpret_cast<uint16_t*>(a.dst)[i] = (uint16_t)(c0 | (c2 << 8)); break;
        case MM_FMT_FP16X4: {
            uint2 o;
            o.x = half_bits((float)c0 / 255.0f) | (half_bits((float)c1 / 255.0f) << 16);
            o.y = half_bits((float)c2 / 255.0f) | (half_bits((float)c3 / 255.0f) << 16);
            reinterpret_cast<uint2*>(a.dst)[i] = o;
            break;
        }
        case MM_FMT_FP8X4: {
            reinterpret_cast<uint32_t*>(a.dst)[i] =
                fp8x4(((float)c0 / 255.0f) * a.inv_scale[0], ((float)c1 / 255.0f) * a.inv_scale[1],
                      ((float)c2 / 255.0f) * a.inv_scale[2], ((float)c3 / 255.0f) * a.inv_scale[3]);
            break;
        }
    }
}

inline unsigned blocks_for(long n) { return (unsigned)((n + 255) / 256); }

// The cells a brick of the volume stages at most (any brick's boxes are within the bound, so what fits it on the
// host fits it in the kernel): the largest layer's; a larger level may still be staged in what others leave.
template <bool HI>
int stage_cap(const GenArgs& a) {
    long cap = 0;
    for (int l0 = 0; l0 < (HI ? kHiLevels : kLowLevels); l0 += HI || l0 ? 3 : 4) {
        long layer = 0;
        for (int l = l0; l < l0 + (HI || l0 ? 3 : 4); l++) {
            const int c = HI ? hi_level_cells(l) : low_level_cells(l), pad = HI || l >= 4 ? 1 : 0;
            layer += box_bound(kBrickX, a.dim, c, pad) * box_bound(kBrickY, a.dim, c, pad) * box_bound(kBrickZ, a.dim, c, pad);
        }
        cap = std::max(cap, layer);
    }
    return (int)std::min<long>(cap, kStageCap);
}
inline long brick_count(const GenArgs& a) {
    return (long)((a.dim + kBrickX - 1) / kBrickX) * ((a.dim + kBrickY - 1) / kBrickY) * ((a.dim + kBrickZ - 1) / kBrickZ);
}

}  // namespace

namespace mm {

size_t noise_workspace_bytes() {
    // gradient table (27^3 B, rounded up) + min/max (6 x u32) + curl field for up to 512^2 texels
    return 20480 + 256 + (size_t)512 * 512 * 3 * sizeof(float);
}

}  // namespace mm

namespace {
// Device scratch of the allocation-free generator entry point: the curl chain's gradient table,
// min/max cells and float curl field for curl maps up to kStaticCurlMax^2 texels. One copy per GPU,
// held until the process ends; every call on that GPU shares it, so calls that overlap on one GPU
// race. The min/max cells are reset by a kernel at the start of every curl generation.
constexpr size_t kScratchBytes = 20480 + 256 + (size_t)MM_STATIC_CURL_MAX * MM_STATIC_CURL_MAX * 3 * sizeof(float);
__device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

namespace mm {

size_t static_scratch_bytes() { return kScratchBytes; }

// The device address of this GPU's copy of `scratch` (the array's name in host code is only a
// stand-in for the symbol), looked up once per device with that device current.
int static_scratch(void** ptr) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return MM_E_DEVICE;
    if (dev < 0 || dev >= kMaxDevices) return MM_E_DEVICE;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return MM_E_DEVICE;
        }
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return MM_OK;
}

namespace {
// A second stream for work that runs beside the caller's (the reprojection beside a phase march): forked from the caller's stream and joined back into it with events, so a call stays ordered on
// that stream and can be captured into a graph. There is one side stream per (device, caller
// stream): a side stream joins whatever capture its caller's stream is in and stays in it until that
// capture ends, so work forked from another caller stream must never reach it. Created on first use
// for each caller stream, up to kMaxSides per process; beyond that the work stays on the caller's
// stream. The caller holds side_lock() from the fork to the join.
struct SideStream {
    int dev = -1;
    hipStream_t main = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};
constexpr int kMaxSides = 256;
std::mutex g_side_mu;
SideStream g_side[kMaxSides];
int g_side_n = 0;

SideStream* side_for(int dev, hipStream_t main) {
    for (int i = 0; i < g_side_n; i++)
        if (g_side[i].dev == dev && g_side[i].main == main) return &g_side[i];
    if (g_side_n == kMaxSides) return nullptr;
    hipStream_t st = nullptr;
    hipEvent_t f = nullptr, j = nullptr;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&f, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&j, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();  // the work then stays on the caller's stream
        if (st) (void)hipStreamDestroy(st);
        if (f) (void)hipEventDestroy(f);
        return nullptr;
    }
    SideStream& d = g_side[g_side_n++];
    d.dev = dev;
    d.main = main;
    d.s = st;
    d.fork = f;
    d.join = j;
    return &d;
}
}  // namespace

std::unique_lock<std::mutex> side_lock() { return std::unique_lock<std::mutex>(g_side_mu); }

hipStream_t side_fork(hipStream_t main) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    SideStream* d = side_for(dev, main);
    if (!d) return nullptr;
    if (hipEventRecord(d->fork, main) != hipSuccess || hipStreamWaitEvent(d->s, d->fork, 0) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return d->s;
}

int side_join(hipStream_t main, hipStream_t side) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return MM_E_DEVICE;
    SideStream* d = side_for(dev, main);
    if (!d || d->s != side) return MM_E_DEVICE;
    if (hipEventRecord(d->join, side) != hipSuccess || hipStreamWaitEvent(main, d->join, 0) != hipSuccess) {
        // the caller's stream could not be ordered after the side work: wait for it here, so nothing
        // the caller enqueues next (such as freeing a workspace the side work reads) overtakes it
        (void)hipGetLastError();
        (void)hipStreamSynchronize(side);
        return MM_E_DEVICE;
    }
    return MM_OK;
}

int launch_generate(const mm_noise_params* p, const mm_noise_set* out, void* workspace, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    auto args = [&](const mm_texture& t, uint32_t seed) {
        return GenArgs{(uint8_t*)t.data, t.width, t.layout == MM_LAYOUT_APRON ? 1 : 0, t.format, seed, p->coverage, {1, 1, 1, 1}};
    };
    Grids g{};
    unsigned blocks = 0;
    size_t lds = 0;
    const bool low128 = (p->what & MM_GEN_LOW_RES) && out->low_res.width == 128;
    if (p->what & MM_GEN_LOW_RES) {
        g.low = args(out->low_res, p->seed);
        if (g.low.fmt == MM_FMT_FP8X4)
            for (int k = 0; k < 4; k++) g.low.inv_scale[k] = 1.0f / out->low_res.scale[k];
        g.lowCap = stage_cap<false>(g.low);
        blocks += low128 ? 128 / k128X * (128 / k128Y) * (128 / k128Z) : (unsigned)brick_count(g.low);
        lds = sizeof(float4) * (low128 ? (size_t)k128LdsCells() : (size_t)g.lowCap);
    }
    if (p->what & MM_GEN_CURL) {
        uint8_t* ws = (uint8_t*)workspace;
        const int dim = out->curl.width;
        g.curl = CurlArgs{ws, (uint32_t*)(ws + 20480), (float*)(ws + 20480 + 256), dim};
        blocks += g.curlBlocks = (dim * dim + kCurlTexels - 1) / kCurlTexels;
        lds = std::max(lds, sizeof(float) * 6 * kCurlTexels);
        hipLaunchKernelGGL(curl_table_kernel, dim3(blocks_for(kLat * kLat * kLat)), dim3(256), 0, s, g.curl.table, g.curl.mm);
    }
    if (p->what & MM_GEN_WEATHER) {
        g.weather = args(out->weather, p->weather_seed);
        const int tiles = (g.weather.dim + kWeatherTile - 1) / kWeatherTile;
        blocks += g.weatherBlocks = tiles * tiles;
        lds = std::max(lds, sizeof(float) * kWeatherCap);
    }
    if (p->what & MM_GEN_HI_RES) {
        g.hi = args(out->hi_res, p->seed);
        g.hiCap = stage_cap<true>(g.hi);
        // beside the low-res volume no more than its blocks' LDS: more would leave fewer of them on a CU (a 9^3
        // hi-res volume's levels of 64 cells would take 54 KB; a 97^3 low-res one needs 30: 196 us against 160)
        if (p->what & MM_GEN_LOW_RES) g.hiCap = std::min(g.hiCap, (int)(lds / sizeof(float4)));
        blocks += g.hiBlocks = (int)brick_count(g.hi);
        lds = std::max(lds, sizeof(float4) * (size_t)g.hiCap);
    }
    if (blocks) hipLaunchKernelGGL(low128 ? maps_kernel<true> : maps_kernel<false>, dim3(blocks), dim3(256), lds, s, g);
    if (p->what & MM_GEN_CURL) {
        const mm_texture& t = out->curl;
        const int dim = t.width, apron = t.layout == MM_LAYOUT_APRON ? 1 : 0;
        const long n = (long)(dim + apron) * (dim + apron);
        hipLaunchKernelGGL(curl_store_kernel, dim3(blocks_for(n)), dim3(256), 0, s, g.curl.field, g.curl.mm, dim, apron,
                           t.format, (uint8_t*)t.data);
    }
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

int launch_pack(int kind, const mm_texture* src, const mm_texture* dst, void* stream) {
    (void)kind;
    PackArgs a;
    a.src = (const uint8_t*)src->data;
    a.dst = (uint8_t*)dst->data;
    a.w = src->width; a.h = src->height; a.d = src->depth;
    a.apron = dst->layout == MM_LAYOUT_APRON ? 1 : 0;
    a.fmt = dst->format;
    a.kind = kind;
    for (int k = 0; k < 4; k++) a.inv_scale[k] = (dst->format == MM_FMT_FP8X4) ? 1.0f / dst->scale[k] : 1.0f;
    const long n = (long)(a.w + a.apron) * (a.h + a.apron) * (a.d > 1 ? a.d + a.apron : 1);
    hipLaunchKernelGGL(pack_kernel, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream, a);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

}  // namespace mm
