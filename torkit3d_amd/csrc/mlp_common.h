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

// A channel's batch norm: (mean, 1 / sqrt(variance + eps), gamma, beta).
__device__ __forceinline__ f32x4 constants_of(const tk3d_mlp_norm &n, int c)
{
    return f32x4{n.mean[c], n.eps < 0.0f ? n.var[c] : 1.0f / __builtin_sqrtf(n.var[c] + n.eps),
                 n.gamma[c], n.beta[c]};
}

// In this order of operations the library's batch norm gives the same bits (a test holds it to that
// on 15 shapes), so that in training the ReLU's signs are those of the forward pass. A scale and a
// shift worked out beforehand would save two operations a value, but round differently.
__device__ __forceinline__ float normalised(float y, f32x4 k)
{
    return __builtin_fmaf(k.z, (y - k.x) * k.y, k.w);
}

// What a pooled layer's backward takes from the activations of a channel in front of it (near their
// mean, include/tk3d_mlp.h).
__device__ __forceinline__ float centre_of(f32x4 k) { return relu(k.w); }

// The sign by which a maximum over relu(norm(y)) becomes one over y.
__device__ __forceinline__ float sign_of(float gamma)
{
    return gamma > 0.0f ? 1.0f : gamma < 0.0f ? -1.0f : 0.0f;
}

// (best, where) or (s, at), the first of the largest; NaN above all.
__device__ __forceinline__ void take_larger(float &best, int &where, float s, int at)
{
    const bool up = s != s ? best == best || at < where : s > best || (s == best && at < where);
    best = up ? s : best;
    where = up ? at : where;
}

// ---- sums and coefficients of a gradient --------------------------------------------------------------

// Sum of (x, y) over the block; the result is valid in every thread.
__device__ __forceinline__ double2 block_sum(double2 v, double2 *lds)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        v.x += __shfl_xor(v.x, off);
        v.y += __shfl_xor(v.y, off);
    }
    const int waves = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0)
        lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double2 s = lds[0];
    for (int w = 1; w < waves; ++w) {
        s.x += lds[w].x;
        s.y += lds[w].y;
    }
    return s;
}

__device__ __forceinline__ double2 slot_sum(const void *partial, int slots, int c, double2 *lds)
{
    const double2 *row = reinterpret_cast<const double2 *>(partial) + (int64_t)c * slots;
    double2 v{0.0, 0.0};
    for (int i = threadIdx.x; i < slots; i += blockDim.x) {
        v.x += row[i].x;
        v.y += row[i].y;
    }
    return block_sum(v, lds);
}

struct Coefficients {
    f32x4 abd;
    float dgamma, dbeta;
};

// (`origin`: the y from which the b y of the caller is counted)
__device__ __forceinline__ Coefficients grad_coefficients(double2 s, double n, const tk3d_mlp_norm &norm,
                                                          int c, double origin = 0.0)
{
    const double is = norm.eps < 0.0f ? (double)norm.var[c]
                                      : 1.0 / __builtin_sqrt((double)norm.var[c] + (double)norm.eps);
    const double gamma = norm.gamma[c], mean = norm.mean[c];
    const double b = -gamma * is * is * is * s.y / n;
    const double d0 = -gamma * is * s.x / n, d = d0 - b * (mean - origin);
    return {f32x4{(float)(gamma * is), (float)b, (float)d, (float)d0}, (float)(s.y * is), (float)s.x};
}

}  // namespace
