// The fp32 functions of one value that elementwise kernels and fused programs
// share, so that both give the same bits (the build disables contraction).
#pragma once

#include <hip/hip_runtime.h>

namespace vchip {

struct ReluOp { __device__ float operator()(float x) const { return x > 0.0f ? x : 0.0f; } };
struct ReluGradOp { __device__ float operator()(float x) const { return x > 0.0f ? 1.0f : 0.0f; } };
struct SigmoidOp {
    // exp(-|x|) cannot overflow: 1 / (1 + e) from 0 up, e / (1 + e) below (src/cpu/cpu_backend.cpp:302-307),
    // without a branch whose two sides a wavefront would run one after the other.
    __device__ static float of(float x, float e) { return (x >= 0.0f ? 1.0f : e) / (1.0f + e); }  // e = exp(-|x|)
    __device__ float operator()(float x) const { return of(x, expf(-fabsf(x))); }
};
struct ExpOp { __device__ float operator()(float x) const { return expf(x); } };
struct LogOp { __device__ float operator()(float x) const { return logf(x); } };

}  // namespace vchip
