// Learned light-cone surrogate: parameter init, feature statistics, BF16 fragment packing, MFMA
// training step (forward, backward, gradient accumulation) and Adam.
//
// The model predicts, for one light-cone job of the march (comp:441-453), the log sun
// transmittance o0 = -D (D = density along the light) and an error bound e = softplus(o1) in
// transmittance units. Loss per sample (T = exp(-D)): (exp(o0) - T)^2 + (e - |exp(o0) - T|)^2, the
// second term with the residual held fixed.
#include <hip/hip_runtime.h>
#include <math.h>
#include <algorithm>
#include "mm_internal.hpp"
#include "surrogate_dev.hpp"
#include "predict_dev.hpp"

using namespace surr;

namespace {

// Model block layout (bytes). All regions 256-byte aligned.
constexpr size_t kPadP = ((kParams * 4 + 255) / 256) * 256;
constexpr size_t offParams = 0, offGrads = kPadP, offM = 2 * kPadP, offV = 3 * kPadP, offStats = 4 * kPadP,
                 offFrags = offStats + 512, offHFrags = offFrags + (size_t)kFrags * 64 * 16,
                 kModelBytes = offHFrags + (size_t)kHFrags * 64 * 16;
// one packing thread per (fragment, lane): the BF16 training fragments, then the FP16 inference ones
constexpr int kPackThreads = (kFrags + kHFrags) * 64;

struct ModelPtrs {
    // grads: nothing reads it (training sums its gradients in buffers of its own); its place keeps the layout of
    // saved blocks, and zeros make a new block the same bytes every time. stats: mean[16], inv_std[16], step, loss
    float *params, *grads, *m, *v, *stats;
    uint4* frags;   // BF16 training fragments (kFrags)
    uint4* hfrags;  // FP16 inference fragments (kHFrags)
};

ModelPtrs ptrs(void* base) {
    uint8_t* b = (uint8_t*)base;
    return ModelPtrs{(float*)(b + offParams), (float*)(b + offGrads), (float*)(b + offM), (float*)(b + offV),
                     (float*)(b + offStats), (uint4*)(b + offFrags), (uint4*)(b + offHFrags)};
}

__device__ __forceinline__ uint32_t hash_u32(uint32_t x) {
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return x;
}

// Glorot-uniform weights, zero biases; Adam state cleared; stats = identity normalisation.
__global__ void init_kernel(float* params, float* m, float* v, float* stats, uint32_t seed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kParams) {
        float w = 0.0f, lim = 0.0f;
        if (i < oB1) lim = sqrtf(6.0f / (kIn + kHidden));
        else if (i >= oW2 && i < oB2) lim = sqrtf(6.0f / (2 * kHidden));
        else if (i >= oW3 && i < oB3) lim = sqrtf(6.0f / (2 * kHidden));
        else if (i >= oW4 && i < oB4) lim = sqrtf(6.0f / (kHidden + kOut));
        if (lim > 0.0f) w = ((hash_u32(seed * 0x9E3779B9u + (uint32_t)i) >> 8) * (1.0f / 16777216.0f) * 2.0f - 1.0f) * lim;
        params[i] = w;
        m[i] = 0.0f;
        v[i] = 0.0f;
    }
    if (i < 16) {
        stats[i] = 0.0f;
        stats[16 + i] = 1.0f;
    }
    if (i >= 32 && i < 64) stats[i] = 0.0f;
}

// Per-feature sums (double) over the sample set, then mean / inverse std.
__global__ void stats_sum_kernel(const float* __restrict__ samples, int n, int stride, double* acc) {
    __shared__ double s[2][kIn][64];
    const int lane = threadIdx.x;
    double sum[kIn], sq[kIn];
    for (int k = 0; k < kIn; k++) sum[k] = sq[k] = 0.0;
    for (long i = (long)blockIdx.x * 64 + lane; i < n; i += (long)gridDim.x * 64) {
        for (int k = 0; k < kIn; k++) {
            double x = samples[i * stride + k];
            sum[k] += x;
            sq[k] += x * x;
        }
    }
    for (int k = 0; k < kIn; k++) { s[0][k][lane] = sum[k]; s[1][k][lane] = sq[k]; }
    __syncthreads();
    if (lane < 2 * kIn) {
        const int w = lane / kIn, k = lane % kIn;
        double t = 0.0;
        for (int j = 0; j < 64; j++) t += s[w][k][j];
        atomicAdd(&acc[w * kIn + k], t);
    }
}

__global__ void stats_final_kernel(const double* acc, int n, float* stats) {
    const int k = threadIdx.x;
    if (k < kIn) {
        double mean = acc[k] / n, var = acc[kIn + k] / n - mean * mean;
        stats[k] = (float)mean;
        stats[16 + k] = (float)(1.0 / sqrt(var > 1e-12 ? var : 1e-12));
    }
}

// FP16 inference fragment element: fragment f, lane half h, column c, element j (k = 8 h + j).
// The inference weights are the training pass's BF16 weights: FP16 holds a BF16 value exactly when
// its magnitude lies in [2^-17, 65504] (8 significant bits; FP16 subnormals keep 8 bits down to
// 2^-17), so the FP16 fragments carry the same weights and only the activations gain precision.
__device__ float bf16_value(float w) { return (float)(__bf16)w; }

__device__ float hfrag_value(const float* __restrict__ p, int f, int h, int c, int j) {
    const int k = 8 * h + j;
    auto bias = [&](int off, int u) {  // k = 0: FP16 b, k = 1: the FP16 rounding of the remainder
        const float b = p[off + u], hi = (float)(_Float16)b;
        return k == 0 ? hi : (k == 1 ? b - hi : 0.0f);
    };
    if (f < kHF2) {
        const int mt = f / 2, u = mt * 32 + c;
        return (f % 2 == 0) ? bias(oB1, u) : bf16_value(p[oW1 + k * kHidden + u]);
    }
    if (f < kHF4) {
        const int base = f < kHF3 ? kHF2 : kHF3, off = f < kHF3 ? oW2 : oW3, boff = f < kHF3 ? oB2 : oB3;
        const int mt = (f - base) / 5, which = (f - base) % 5, u = mt * 32 + c;
        return which == 0 ? bias(boff, u) : bf16_value(p[off + kperm(which - 1, h, j) * kHidden + u]);
    }
    const int kt = f - kHF4;
    return c < kOut ? bf16_value(p[oW4 + kperm(kt, h, j) * kOut + c]) : 0.0f;
}

// BF16 A-operand fragments (see surrogate_dev.hpp), then the FP16 inference fragments. One thread per
// (fragment, lane).
__global__ void pack_kernel(const float* __restrict__ p, uint4* __restrict__ frags, uint4* __restrict__ hfrags) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= kPackThreads) return;
    if (t >= kFrags * 64) {
        const int ti = t - kFrags * 64, f = ti / 64, lane = ti % 64;
        f16x8 r;
        for (int j = 0; j < 8; j++) r[j] = (_Float16)hfrag_value(p, f, lane >> 5, lane & 31, j);
        hfrags[ti] = __builtin_bit_cast(uint4, r);
        return;
    }
    const int frag = t / 64, lane = t % 64, h = lane >> 5, c = lane & 31;
    float v[8];
    for (int j = 0; j < 8; j++) {
        float w = 0.0f;
        if (frag < kFragF2) {                        // forward L1: W1[k][u], k = 8h + j, u = mt*32 + c
            const int mt = frag - kFragF1;
            w = p[oW1 + (8 * h + j) * kHidden + mt * 32 + c];
        } else if (frag < kFragF4) {                 // forward L2/L3: W[k = kperm][u]
            const int base = frag < kFragF3 ? kFragF2 : kFragF3, off = frag < kFragF3 ? oW2 : oW3;
            const int mt = (frag - base) / 4, kt = (frag - base) % 4;
            w = p[off + kperm(kt, h, j) * kHidden + mt * 32 + c];
        } else if (frag < kFragB4) {                 // forward L4: W4[k = kperm][u = c] for u < 2
            const int kt = frag - kFragF4;
            w = c < kOut ? p[oW4 + kperm(kt, h, j) * kOut + c] : 0.0f;
        } else if (frag < kFragB3) {                 // backward L4: A[u3 = mt*32 + c][k = out 8h + j]
            const int mt = frag - kFragB4, k = 8 * h + j;
            w = k < kOut ? p[oW4 + (mt * 32 + c) * kOut + k] : 0.0f;
        } else {                                     // backward L3/L2: A[u_in = mt*32 + c][k = kperm(u_out)]
            const int base = frag < kFragB2 ? kFragB3 : kFragB2, off = frag < kFragB2 ? oW3 : oW2;
            const int mt = (frag - base) / 4, kt = (frag - base) % 4;
            w = p[off + (mt * 32 + c) * kHidden + kperm(kt, h, j)];
        }
        v[j] = w;
    }
    bf16x8 b = pack8(v);
    frags[t] = __builtin_bit_cast(uint4, b);
}

// ---------------------------------------------------------------- training
// Gradients of a batch: a block of four waves takes 128 rows, 32 per wave. Each wave runs its rows' forward
// and backward passes in registers (pre-activations included: one wave per SIMD may use them all) and leaves
// the activations and dZ of every layer in LDS, transposed to [unit][row] in BF16. After one barrier the
// four waves share the weight gradients dW^T = dZ^T a^T, a 32x32 tile of dW2 and of dW3 and two of the smaller
// tiles each, over all 128 rows, in MFMA accumulators that persist over the blocks of rows a workgroup takes.
// The bias gradients are products with ones (dW1's 17th column; tiles of their own for layers 2 and 3).
//
// A step is bound by latency, not by its 15 MFLOP: 64 workgroups at the configured batch, each a chain of about
// 75 MFMAs per wave. One wave per 64 rows with the gradients added by atomics from every 32-row tile (2.4 M
// device-scope atomics a step) and separate clearing, Adam and packing launches took 146 us a step; this takes
// 11.5 us and the update 4. The gradient of a million rows: 12.5 ms before, 0.16 ms
// (0.26 with the workgroups' atomics in MFMA order, a cache line each, instead of through LDS; of 30 000 rows 112
// us against 24). The weights go through LDS once
// per workgroup: each wave loading its own fragments into registers took 15.7 us (144 of them, the rest in
// accumulator registers at a move per use).
constexpr int kTrainRows = 128, kTrainWaves = kTrainRows / 32;
constexpr int kRowPitch = kTrainRows + 8;  // 16 bytes of padding: the 32 lanes' 16-byte reads spread over the banks
constexpr int kMaxTrainBlocks = 256;       // one per CU; larger batches loop
constexpr int kPartial = (kParams + 1 + 15) / 16 * 16;  // a workgroup's gradients and loss, floats
static_assert(kTrainWaves == 4 && kFrags % kTrainWaves == 0, "the tiles' split");

struct alignas(16) TrainLds {
    __bf16 act[3][kHidden][kRowPitch];  // activations of layers 1 to 3
    __bf16 dz[3][kHidden][kRowPitch];
    __bf16 x[32][kRowPitch];            // inputs; row 16 is ones, the rest unused
    __bf16 dz4[kOut][kRowPitch];
    uint4 frag[kFrags * 64];            // the weights, loaded once for the four waves
    float bias[3][kHidden];
    float red[kTrainWaves][3];
};

__device__ __forceinline__ void put4(float* g, int i, const f32x16& a, int r) {  // i a multiple of 4
    *reinterpret_cast<float4*>(g + i) = make_float4(a[r], a[r + 1], a[r + 2], a[r + 3]);
}

// Rows: hashed draws from the n samples (`rows` = the batch) by the model's step counter plus `step`, or, with
// no counter, samples 0 .. n - 1 (rows = n).
// out: ATOMIC ? the gradients, with the loss at `loss` : the partial buffers, the loss at [kParams].
template <bool ATOMIC>
__global__ __launch_bounds__(64 * kTrainWaves, 1) void train_kernel(
    const float* __restrict__ samples, int n, int stride, const float* __restrict__ params,
    const float* __restrict__ stats, const uint4* __restrict__ frags, float* __restrict__ out,
    float* __restrict__ loss, uint32_t seed, const int* __restrict__ counter, int step, int rows, float invB) {
    __shared__ TrainLds L;
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = 32 * w + c;  // this lane's row within the block
    float mean[8], inv[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        mean[j] = stats[8 * h + j];
        inv[j] = stats[16 + 8 * h + j];
    }
    const uint32_t draw = counter ? (uint32_t)(*counter + step) * 0x632BE5ABu : 0u;
    // this lane's half of its row's features and the row's D, fetched ahead of the rows in work
    float next[9];
    auto fetch = [&](int b) {
        const uint32_t row = (uint32_t)b * kTrainRows + (uint32_t)col;
        uint32_t idx = row < (uint32_t)rows ? row : 0u;
        if (counter) idx = hash_u32(seed ^ hash_u32(draw + row)) % (uint32_t)n;
        const float* src = samples + (size_t)idx * stride;
#pragma unroll
        for (int j = 0; j < 8; j++) next[j] = src[8 * h + j];
        next[8] = src[kIn];
    };
    const int blocks = (rows + kTrainRows - 1) / kTrainRows;
    fetch(blockIdx.x);
#pragma unroll
    for (int k = 0; k < kFrags / kTrainWaves; k++)
        L.frag[64 * kTrainWaves * k + threadIdx.x] = frags[64 * kTrainWaves * k + threadIdx.x];
    if (threadIdx.x < 3 * kHidden) {
        const int l = threadIdx.x / kHidden, u = threadIdx.x % kHidden;
        L.bias[l][u] = params[(l == 0 ? oB1 : l == 1 ? oB2 : oB3) + u];
    }
    auto frag = [&](int k) { return __builtin_bit_cast(bf16x8, L.frag[64 * k + lane]); };
    if (h == 0) L.x[kIn][col] = (__bf16)1.0f;
    __syncthreads();
    f32x16 acc[4] = {};
    float lossv = 0.0f, db4[2] = {0.0f, 0.0f};
    for (int b = blockIdx.x; b < blocks; b += gridDim.x) {
        const bool valid = (uint32_t)b * kTrainRows + (uint32_t)col < (uint32_t)rows;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = (next[j] - mean[j]) * inv[j];
        const float T = __expf(-next[8]);
        if (b + (int)gridDim.x < blocks) fetch(b + (int)gridDim.x);
        const bf16x8 xb = pack8(x);
#pragma unroll
        for (int j = 0; j < 8; j++) L.x[8 * h + j][col] = xb[j];
        // ---- forward: pre-activations z stay in registers, activations go to LDS
        float z[3][32];
        bf16x8 a[4];
#pragma unroll
        for (int l = 0; l < 3; l++) {
            f32x16 t[2];  // accumulators start at the biases
#pragma unroll
            for (int r = 0; r < 32; r++) t[r / 16][r % 16] = L.bias[l][(r / 16) * 32 + crow(r % 16, h)];
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                if (l == 0) t[mt] = mfma(frag(kFragF1 + mt), xb, t[mt]);
                else
                    for (int kt = 0; kt < 4; kt++)
                        t[mt] = mfma(frag((l == 1 ? kFragF2 : kFragF3) + mt * 4 + kt), a[kt], t[mt]);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                float v[16];
                for (int r = 0; r < 16; r++) {
                    z[l][mt * 16 + r] = t[mt][r];
                    v[r] = hswish(t[mt][r]);
                }
                a[2 * mt] = pack8(v);
                a[2 * mt + 1] = pack8(v + 8);
            }
#pragma unroll
            for (int r = 0; r < 32; r++) L.act[l][(r / 16) * 32 + crow(r % 16, h)][col] = a[r / 8][r % 8];
        }
        // ---- output layer, loss and dZ4 (the outputs of row c are in the lanes of half 0)
        f32x16 o = {};
#pragma unroll
        for (int kt = 0; kt < 4; kt++) o = mfma(frag(kFragF4 + kt), a[kt], o);
        float dz4[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (h == 0) {
            const float o0 = o[0] + params[oB4], o1 = o[1] + params[oB4 + 1];
            const float p = __expf(o0), r = p - T, ar = fabsf(r);
            const float e = softplus(o1), sig = 1.0f / (1.0f + __expf(-o1));
            if (valid) {
                lossv += r * r + (e - ar) * (e - ar);
                dz4[0] = (2.0f * r * p) * invB;
                dz4[1] = (2.0f * (e - ar) * sig) * invB;
            }
        }
        const bf16x8 d4 = pack8(dz4);
        if (h == 0) {
            L.dz4[0][col] = d4[0];
            L.dz4[1][col] = d4[1];
            db4[0] += (float)d4[0];
            db4[1] += (float)d4[1];
        }
        // ---- backward: dA = W dZ (dZ in registers as the B operand, k permuted), dZ = dA hswish'(z)
#pragma unroll
        for (int l = 2; l >= 0; l--) {
            f32x16 t[2] = {};
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                if (l == 2) t[mt] = mfma(frag(kFragB4 + mt), d4, t[mt]);
                else
                    for (int kt = 0; kt < 4; kt++)
                        t[mt] = mfma(frag((l == 1 ? kFragB3 : kFragB2) + mt * 4 + kt), a[kt], t[mt]);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                float v[16];
                for (int r = 0; r < 16; r++) v[r] = t[mt][r] * hswish_grad(z[l][mt * 16 + r]);
                a[2 * mt] = pack8(v);
                a[2 * mt + 1] = pack8(v + 8);
            }
#pragma unroll
            for (int r = 0; r < 32; r++) L.dz[l][(r / 16) * 32 + crow(r % 16, h)][col] = a[r / 8][r % 8];
        }
        __syncthreads();
        // ---- weight gradients: M = units (rows of dZ^T), N = inputs (rows of a^T), K = the block's rows
        // wave w: tile (w / 2, w % 2) of dW3 and dW2; waves 0, 1: dW1 and db1 (the inputs with their row of ones), db2;
        // waves 2, 3: db3 (products with ones), dW4
        const int mt = w >> 1, nt = w & 1;
        const bool lower = w < 2;
        const __bf16* A[4] = {L.dz[2][32 * mt + c], L.dz[1][32 * mt + c], L.dz[lower ? 0 : 2][32 * nt + c],
                              lower ? L.dz[1][32 * nt + c] : L.dz4[c & 1]};
        const __bf16* B[4] = {L.act[1][32 * nt + c], L.act[0][32 * nt + c], L.x[lower ? c : kIn],
                              lower ? L.x[kIn] : L.act[2][32 * nt + c]};
#pragma unroll
        for (int kt = 0; kt < kTrainRows / 16; kt++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = 16 * kt + 8 * h;
                acc[q] = mfma(*reinterpret_cast<const bf16x8*>(A[q] + k), *reinterpret_cast<const bf16x8*>(B[q] + k),
                              acc[q]);
            }
        __syncthreads();  // the next rows overwrite the tiles
    }
    // ATOMIC: put together in LDS (the tiles are no longer read), then added in order, 64 neighbours at a time
    static_assert(sizeof(TrainLds::act) >= sizeof(float) * kPartial, "the gradients take the activations' place");
    float* g = ATOMIC ? reinterpret_cast<float*>(&L.act) : out + (size_t)blockIdx.x * kPartial;
    // loss and output biases: summed over the wave, then over the four waves
    for (int off = 32; off > 0; off >>= 1) {
        lossv += __shfl_xor(lossv, off);
        db4[0] += __shfl_xor(db4[0], off);
        db4[1] += __shfl_xor(db4[1], off);
    }
    if (lane == 0) {
        L.red[w][0] = lossv;
        L.red[w][1] = db4[0];
        L.red[w][2] = db4[1];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        float s = 0.0f;
        for (int k = 0; k < kTrainWaves; k++) s += L.red[k][threadIdx.x];
        g[threadIdx.x == 0 ? kParams : oB4 + (int)threadIdx.x - 1] = s;
    }
    const int mt = w >> 1, nt = w & 1;
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
        const int u = 2 * r + 4 * h;  // crow(r, h)
        put4(g, oW3 + (32 * nt + c) * kHidden + 32 * mt + u, acc[0], r);
        put4(g, oW2 + (32 * nt + c) * kHidden + 32 * mt + u, acc[1], r);
        if (w < 2) {
            if (c < kIn) put4(g, oW1 + c * kHidden + 32 * nt + u, acc[2], r);
            if (c == kIn) put4(g, oB1 + 32 * nt + u, acc[2], r);
            if (c == 0) put4(g, oB2 + 32 * nt + u, acc[3], r);
        } else if (c == 0) {
            put4(g, oB3 + 32 * nt + u, acc[2], r);
        }
    }
    if (w >= 2 && h == 0) {
        g[oW4 + (32 * nt + c) * kOut] = acc[3][0];
        g[oW4 + (32 * nt + c) * kOut + 1] = acc[3][1];
    }
    if constexpr (ATOMIC) {
        __syncthreads();
        for (int i = (int)threadIdx.x; i <= kParams; i += 64 * kTrainWaves) atomicAdd(i < kParams ? out + i : loss, g[i]);
    }
}

// Where parameter i enters the packed fragments (the inverse of pack_kernel's maps), written there.
__device__ __forceinline__ void kperm_inverse(int k, int& kt, int& h, int& j) {
    kt = (k / 32) * 2 + (k % 32) / 16;
    h = (k / 4) % 2;
    j = ((k % 16) / 8) * 4 + k % 4;
}
__device__ void scatter_param(int i, float p, uint4* frags, uint4* hfrags) {
    __bf16* fb = reinterpret_cast<__bf16*>(frags);
    _Float16* fh = reinterpret_cast<_Float16*>(hfrags);
    auto slot = [](int frag, int h, int c, int j) { return (frag * 64 + h * 32 + c) * 8 + j; };
    const float bw = bf16_value(p);
    auto bias = [&](int frag, int u) {
        const float hi = (float)(_Float16)p;
        fh[slot(frag, 0, u % 32, 0)] = (_Float16)hi;
        fh[slot(frag, 0, u % 32, 1)] = (_Float16)(p - hi);
    };
    int kt, h, j;
    if (i < oB1) {
        const int k = i / kHidden, u = i % kHidden;
        fb[slot(kFragF1 + u / 32, k / 8, u % 32, k % 8)] = (__bf16)p;
        fh[slot(kHF1 + 2 * (u / 32) + 1, k / 8, u % 32, k % 8)] = (_Float16)bw;
    } else if (i < oW2) {
        bias(kHF1 + 2 * ((i - oB1) / 32), i - oB1);
    } else if (i < oW4) {
        const bool two = i < oW3;
        const int e = i - (two ? oW2 : oW3), hf = two ? kHF2 : kHF3;
        if (e >= kHidden * kHidden) {
            const int u = e - kHidden * kHidden;
            bias(hf + 5 * (u / 32), u);
        } else {
            const int k = e / kHidden, u = e % kHidden;
            kperm_inverse(k, kt, h, j);
            fb[slot((two ? kFragF2 : kFragF3) + (u / 32) * 4 + kt, h, u % 32, j)] = (__bf16)p;
            fh[slot(hf + 5 * (u / 32) + 1 + kt, h, u % 32, j)] = (_Float16)bw;
            kperm_inverse(u, kt, h, j);
            fb[slot((two ? kFragB2 : kFragB3) + (k / 32) * 4 + kt, h, k % 32, j)] = (__bf16)p;
        }
    } else if (i < oB4) {
        const int k = (i - oW4) / kOut, o = (i - oW4) % kOut;
        kperm_inverse(k, kt, h, j);
        fb[slot(kFragF4 + kt, h, o, j)] = (__bf16)p;
        fh[slot(kHF4 + kt, h, o, j)] = (_Float16)bw;
        fb[slot(kFragB4 + k / 32, 0, k % 32, o)] = (__bf16)p;
    }
}

// One Adam update from the workgroups' partial gradients: a block takes 64 parameters, each summed by 4
// threads (every fourth partial) in a fixed order; the first of them updates the parameter, its moments
// and its places in the packed fragments. Parameter kParams is the loss. One launch in place of a
// reduction, Adam, a repack of all 4096 fragment lanes and the clearing of the gradients.
__global__ __launch_bounds__(256) void update_kernel(const float* __restrict__ part, int nb, float* params, float* m,
                                                     float* v, uint4* frags, uint4* hfrags, float* loss, float lr,
                                                     float b1, float b2, float eps, const int* __restrict__ counter,
                                                     int step) {
    __shared__ float sum[4][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    float s = 0.0f;
    if (i <= kParams) {
#pragma unroll 8
        for (int b = grp; b < nb; b += 4) s += part[(size_t)b * kPartial + i];
    }
    sum[grp][lane] = s;
    __syncthreads();
    if (grp != 0 || i > kParams) return;
    const float g = (sum[0][lane] + sum[1][lane]) + (sum[2][lane] + sum[3][lane]);
    if (i == kParams) {
        *loss = g;
        return;
    }
    const int t = *counter + step + 1;
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / (1.0f - powf(b1, (float)t)), vh = vi / (1.0f - powf(b2, (float)t));
    const float p = params[i] - lr * mh / (sqrtf(vh) + eps);
    params[i] = p;
    scatter_param(i, p, frags, hfrags);
}

__global__ void advance_kernel(int* counter, int steps) { *counter += steps; }

__global__ void zero_kernel(float* p, int n, float* one) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
    if (i == 0 && one) *one = 0.0f;
}

inline unsigned blocks(long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

namespace mm {

size_t surrogate_model_bytes() { return kModelBytes; }

int surrogate_init(void* model, uint32_t seed, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    ModelPtrs p = ptrs(model);
    hipLaunchKernelGGL(init_kernel, dim3(blocks(kParams, 256)), dim3(256), 0, s, p.params, p.m, p.v, p.stats, seed);
    hipLaunchKernelGGL(zero_kernel, dim3(blocks(kParams, 256)), dim3(256), 0, s, p.grads, kParams, nullptr);
    hipLaunchKernelGGL(pack_kernel, dim3(blocks(kPackThreads, 256)), dim3(256), 0, s, p.params, p.frags, p.hfrags);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

int surrogate_fit_stats(void* model, const float* samples, int n, int stride, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    ModelPtrs p = ptrs(model);
    double* acc = nullptr;
    if (hipMallocAsync((void**)&acc, sizeof(double) * 2 * kIn, s) != hipSuccess) return MM_E_DEVICE;
    hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(64), 0, s, (float*)acc, 4 * kIn, nullptr);
    hipLaunchKernelGGL(stats_sum_kernel, dim3(256), dim3(64), 0, s, samples, n, stride, acc);
    hipLaunchKernelGGL(stats_final_kernel, dim3(1), dim3(64), 0, s, acc, n, p.stats);
    (void)hipFreeAsync(acc, s);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

int surrogate_train(void* model, const float* samples, int n, int stride, int batch, int steps, float lr,
                    uint32_t seed, float* loss_out, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    ModelPtrs p = ptrs(model);
    int* counter = reinterpret_cast<int*>(p.stats + 32);  // Adam steps taken; stays on the device
    const int nb = std::min(kMaxTrainBlocks, (batch + kTrainRows - 1) / kTrainRows);
    float* part = nullptr;  // the workgroups' partial gradients, for this call
    if (steps > 0 && hipMallocAsync((void**)&part, sizeof(float) * (size_t)nb * kPartial, s) != hipSuccess)
        return MM_E_DEVICE;
    for (int i = 0; i < steps; i++) {
        hipLaunchKernelGGL(train_kernel<false>, dim3(nb), dim3(64 * kTrainWaves), 0, s, samples, n, stride, p.params,
                           p.stats, p.frags, part, nullptr, seed, counter, i, batch, 1.0f / (float)batch);
        hipLaunchKernelGGL(update_kernel, dim3(blocks(kParams + 1, 64)), dim3(256), 0, s, part, nb, p.params, p.m, p.v,
                           p.frags, p.hfrags, loss_out ? loss_out + i : p.stats + 33, lr, 0.9f, 0.999f, 1e-8f, counter,
                           i);
    }
    hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(1), 0, s, counter, steps);
    const int e = hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
    if (part) (void)hipFreeAsync(part, s);
    return hipStreamSynchronize(s) == hipSuccess ? e : MM_E_DEVICE;
}

int surrogate_load(void* model, const float* params, const float* stats, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    ModelPtrs p = ptrs(model);
    if (params && hipMemcpyAsync(p.params, params, sizeof(float) * kParams, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return MM_E_DEVICE;
    if (stats && hipMemcpyAsync(p.stats, stats, sizeof(float) * 2 * kIn, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return MM_E_DEVICE;
    hipLaunchKernelGGL(pack_kernel, dim3(blocks(kPackThreads, 256)), dim3(256), 0, s, p.params, p.frags, p.hfrags);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

int surrogate_gradient(const void* model, const float* samples, int n, int stride, float* grad_out, float* loss_out,
                       void* stream) {
    hipStream_t s = (hipStream_t)stream;
    ModelPtrs p = ptrs(const_cast<void*>(model));
    hipLaunchKernelGGL(zero_kernel, dim3(blocks(kParams, 256)), dim3(256), 0, s, grad_out, kParams, loss_out);
    const unsigned nb = std::min(blocks(n, kTrainRows), (unsigned)kMaxTrainBlocks);
    hipLaunchKernelGGL(train_kernel<true>, dim3(nb), dim3(64 * kTrainWaves), 0, s, samples, n, stride, p.params,
                       p.stats, p.frags, grad_out, loss_out, 0u, nullptr, 0, n, 1.0f / (float)n);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

// Prediction with this file's MFMA form (see predict.hip for when).
int surrogate_predict_few(const void* model, const float* x, int n, int stride, float* out, void* stream) {
    return launch_predict(model, x, n, stride, out, stream);
}

const float* surrogate_params(const void* model) { return ptrs(const_cast<void*>(model)).params; }
const float* surrogate_stats(const void* model) { return ptrs(const_cast<void*>(model)).stats; }
const uint4* surrogate_frags(const void* model) { return ptrs(const_cast<void*>(model)).frags; }
const uint4* surrogate_infer_frags(const void* model) { return ptrs(const_cast<void*>(model)).hfrags; }

}  // namespace mm
