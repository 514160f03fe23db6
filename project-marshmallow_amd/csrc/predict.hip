// Batch prediction of the learned light-cone surrogate, and the choice of its kernel's form (predict_dev.hpp).
#include <hip/hip_runtime.h>
#include "predict_dev.hpp"

namespace mm {

// Ordinary registers while their five waves a SIMD (1024 SIMDs, 64 rows a wave: 327 680 rows) take the rows at once
// or nearly so, the accumulator file beyond. us, ordinary / accumulator file: 1000 rows 5.3 / 6.1, 100 000 7.1 / 7.7,
// 300 000 20.4 / 23.3, 327 680 22.1 / 24.3, 348 000 24.8 / 24.8; 360 000 25.9 / 25.3, 400 000 28.4 / 27.4, 500 000
// 34.6 / 32.3, 800 000 50.4 / 51.5, 1 M 61.0 / 61.2, 2 M 112.8 / 111.6, 4 M 233 / 229.
constexpr int kFewRows = 348000;

int surrogate_predict(const void* model, const float* x, int n, int stride, float* out, void* stream) {
    return n <= kFewRows ? surrogate_predict_few(model, x, n, stride, out, stream)
                              : launch_predict(model, x, n, stride, out, stream);
}

}  // namespace mm
