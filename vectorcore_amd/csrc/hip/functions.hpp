// The fp32 functions of one value that elementwise kernels and fused programs
// share, so that both give the same bits (the build disables contraction).
#pragma once

#include <hip/hip_runtime.h>

namespace vchip {

struct ReluOp { __device__ float operator()(float x) const { return x > 0.0f ? x : 0.0f; } };
struct ReluGradOp { __device__ float operator()(float x) const { return x > 0.0f ? 1.0f : 0.0f; } };
struct SigmoidOp {
    // The branch keeps exp() from overflowing (src/cpu/cpu_backend.cpp:302-307).
    __device__ float operator()(float x) const {
        if (x >= 0.0f) return 1.0f / (1.0f + expf(-x));
        const float e = expf(x);
        return e / (1.0f + e);
    }
};
struct ExpOp { __device__ float operator()(float x) const { return expf(x); } };
struct LogOp { __device__ float operator()(float x) const { return logf(x); } };

}  // namespace vchip
