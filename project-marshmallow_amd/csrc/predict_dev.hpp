// Batch prediction's kernel, included by two translation units that are built with different MFMA forms:
// surrogate.hip keeps the accumulators in ordinary registers (643 instructions, 91 registers: five waves a SIMD),
// predict.hip leaves them to the accumulator file (777, four waves). Same operations, same results.
#pragma once
#include "mm_internal.hpp"
#include "surrogate_dev.hpp"

namespace {

using namespace surr;

// Batch inference with the march's FP16 path: 64 samples per wave; out[i] = (o0, softplus(o1)).
__global__ __launch_bounds__(64) void predict_kernel(const float* __restrict__ x, int n, int stride,
                                                     const float* __restrict__ params, const float* __restrict__ stats,
                                                     const uint4* __restrict__ hfrags, float* __restrict__ out) {
    const int lane = threadIdx.x;
    const long i = (long)blockIdx.x * 64 + lane;
    float f[kIn];
    for (int k = 0; k < kIn; k++) f[k] = i < n ? (x[i * stride + k] - stats[k]) * stats[16 + k] : 0.0f;
    const long left = (long)n - (long)blockIdx.x * 64;
    FwdOut o = mlp_infer64_h(hfrags, params + oB4, f, left < 64 ? (int)left : 64);
    if (i < n) {
        out[i * 2 + 0] = o.o0;
        out[i * 2 + 1] = softplus(o.o1);
    }
}

inline int launch_predict(const void* model, const float* x, int n, int stride, float* out, void* stream) {
    const unsigned blocks = (unsigned)(((long)n + 63) / 64);
    hipLaunchKernelGGL(predict_kernel, dim3(blocks), dim3(64), 0, (hipStream_t)stream, x, n, stride,
                       mm::surrogate_params(model), mm::surrogate_stats(model), mm::surrogate_infer_frags(model), out);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

}  // namespace
