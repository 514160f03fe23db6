// Checks cr_math.hpp's conversions on the GPU over float bit patterns [lo, hi).
//   miss[0]  fp8_pair against the FP8 e4m3 rounding written out, in each of the four bytes
//   miss[1]  floor_half_up against floor of v + 0.5 rounded to float, for the coordinates of the post chain's taps:
//            0 <= v <= 2^22 and a multiple of 2^-17
#include <hip/hip_runtime.h>
#include "../../project-marshmallow_amd/csrc/cr_math.hpp"

__device__ unsigned fp8_written_out(float v) {
    if (!(v > 0.0f)) return 0u;
    if (v >= 448.0f) return 0x7Eu;
    const unsigned u = __float_as_uint(v);
    const int e = (int)(u >> 23) - 127;
    if (e < -6) return (unsigned)rintf(v * 512.0f);  // subnormal: multiples of 2^-9; 8 is the smallest normal
    unsigned code = ((unsigned)(e + 7) << 3) | ((u >> 20) & 7u);
    const unsigned rest = u & 0xfffffu;
    if (rest > 0x80000u || (rest == 0x80000u && (code & 1u))) code++;  // carries into the exponent
    return code > 0x7Eu ? 0x7Eu : code;
}

__global__ void cvt_check_kernel(unsigned lo, unsigned hi, unsigned long long* miss) {
    unsigned long long fp8 = 0, half = 0;
    const unsigned long long step = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long u = lo + (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; u <= hi; u += step) {
        const float v = __uint_as_float((unsigned)u);
        const unsigned want = fp8_written_out(v), all = want | want << 8 | want << 16 | want << 24;
        fp8 += fp8_pair<true>(v, v, fp8_pair<false>(v, v, 0u)) != all;
        if (v >= 0.0f && v <= 0x1p22f && v * 0x1p17f == floorf(v * 0x1p17f))
            half += floor_half_up(v) != (int)floorf(v + 0.5f);
    }
    if (fp8) atomicAdd(&miss[0], fp8);
    if (half) atomicAdd(&miss[1], half);
}

extern "C" int mm_cvt_check(unsigned lo, unsigned hi, unsigned long long* miss, void* stream) {
    hipLaunchKernelGGL(cvt_check_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, lo, hi, miss);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
