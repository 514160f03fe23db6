// Checks cr_math.hpp's square root and reciprocals on the GPU: mm_rn_check counts, over the float bit patterns
// [lo, hi), the results of the device forms that differ from the correctly rounded ones (from FP64, whose
// square root and quotient of a float round to the same float).
#include <hip/hip_runtime.h>
#include "../../project-marshmallow_amd/csrc/cr_math.hpp"

__global__ void rn_check_kernel(unsigned lo, unsigned hi, unsigned long long* miss) {
    unsigned long long root = 0, inv = 0, rcp = 0;
    const unsigned long long step = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long u = lo + (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; u < hi; u += step) {
        const float x = __uint_as_float((unsigned)u);
        const float s = (float)sqrt((double)x);
        root += sqrt_rn_rsq(x) != s;
        inv += rcp_sqrt_rn(x) != (float)(1.0 / (double)s);
        rcp += rcp_rn(x) != (float)(1.0 / (double)x);
    }
    if (root) atomicAdd(&miss[0], root);
    if (inv) atomicAdd(&miss[1], inv);
    if (rcp) atomicAdd(&miss[2], rcp);
}

extern "C" int mm_rn_check(unsigned lo, unsigned hi, unsigned long long* miss, void* stream) {
    hipLaunchKernelGGL(rn_check_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, lo, hi, miss);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
