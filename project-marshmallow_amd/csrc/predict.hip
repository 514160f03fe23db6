// Batch prediction of the learned light-cone surrogate: a translation unit of its own, without the flag that keeps
// the training kernel's MFMA accumulators in ordinary registers. With it this kernel takes 91 registers, all
// ordinary, and 500 000 rows 36.5 us; without it, accumulators in the accumulator file, 34.4 us.
#include <hip/hip_runtime.h>
#include "mm_internal.hpp"
#include "surrogate_dev.hpp"

using namespace surr;

namespace {

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

}  // namespace

namespace mm {

int surrogate_predict(const void* model, const float* x, int n, int stride, float* out, void* stream) {
    const unsigned blocks = (unsigned)(((long)n + 63) / 64);
    hipLaunchKernelGGL(predict_kernel, dim3(blocks), dim3(64), 0, (hipStream_t)stream, x, n, stride,
                       surrogate_params(model), surrogate_stats(model), surrogate_infer_frags(model), out);
    return hipGetLastError() == hipSuccess ? MM_OK : MM_E_DEVICE;
}

}  // namespace mm
