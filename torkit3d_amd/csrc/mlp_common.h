// Device helpers of the shared-MLP kernels (mlp.hip, edge_conv.hip).
#pragma once

#include "tk3d_common.h"
#include "tk3d_mlp.h"

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / TK_WAVE;

// ReLU that keeps NaN, as torch's does.
__device__ __forceinline__ float relu(float z) { return __builtin_elementwise_maximum(z, 0.0f); }
// Whether the gradient passes a ReLU whose input was z (torch: where the output is > 0 or NaN).
__device__ __forceinline__ bool passes(float z) { return !(z <= 0.0f); }

__device__ __forceinline__ f32x2 scale_shift(const tk3d_mlp_norm &n, int c)
{
    const float scale = n.gamma[c] * (1.0f / __builtin_sqrtf(n.var[c] + n.eps));
    return f32x2{scale, __builtin_fmaf(-n.mean[c], scale, n.beta[c])};
}

// The sign by which a maximum over relu(norm(y)) becomes one over y.
__device__ __forceinline__ float sign_of(float gamma)
{
    return gamma > 0.0f ? 1.0f : gamma < 0.0f ? -1.0f : 0.0f;
}

}  // namespace
