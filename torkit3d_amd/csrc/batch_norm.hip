// Batch norm of a training step's forward pass with its ReLU, or its ReLU and maximum over groups.
//
// The activations of a training step are the library's bit by bit (native_mlp.cpp says why), so the
// sums here come in the order in which its batch norm adds them up. That order was found from its
// results alone: with 2^45 at one position, -2^45 at another and ones elsewhere, the sum counts the
// values that are added after the two have met (the method of FPRev, Xie et al. 2025), and the
// rounding of mean, 1 / sqrt(variance + eps) and the running statistics left one formula each. For rows
// of P values, P % 4 == 0, the batch's rows behind one another:
//   P >= 4096         thread t of 1024 takes values 4 t .. 4 t + 3, 4 t + 4096 .. and so on
//   1024 < P < 4096   thread t takes values t, t + 1024, ...
// one value after the other (fma for the squares); 64 consecutive threads are added up as a binary
// tree, the sixteen results in order. Other rows, and batches for which it takes other kernels, are
// left to it (tk3d_mlp_batch_norm_supported).
//
// What bounds it: memory. The library takes one workgroup per channel, 64 of them on 256 CUs, that
// reads the values twice and writes them, a ReLU that reads and writes them again, and the maximum a
// fourth time. The thread chains of a channel do not depend on each other, so here a wave of their own
// (16 per channel) runs 64 of them, sixteen loads ahead; the second kernel reads the values again, partly
// from the last-level cache, normalises and writes or keeps maxima alone. Measured (us, the library alone
// -> the two kernels with ReLU, or with maximum): [16, 64, 512, 32] 110 -> 35, 33; [16, 128, 128, 64] 59
// -> 33, 32; [8, 32, 2048, 32] 214 -> 37, 34; [8, 128, 16384] 59 -> 32; [8, 1024, 2048] 34 -> 34; [8, 64,
// 2048, 20] 138 -> 40, 31 (84 MB: sums 14.6 us, 5.7 TB/s). The ReLU (10 to 14 us) and the maximum (40 to
// 57 us) that the library needed behind it come on top of its times. Every workgroup of the second adds up the
// sixteen results of its channel itself.
#include "mlp_common.h"

namespace {

constexpr int kLibraryWaves = 16;  // of 64 threads each
constexpr int kAhead = 16;         // loads in flight per lane

// The sums of 64 of a channel's 1024 chains; V consecutive values at a time.
template <int V>
__global__ void __launch_bounds__(kBlock) batch_sums_kernel(const float *__restrict__ y, int B, int C,
                                                            int P, float2 *__restrict__ partial)
{
    typedef float vec __attribute__((ext_vector_type(V)));
    constexpr int STEP = kLibraryWaves * TK_WAVE * V;
    const int c = blockIdx.x / (kLibraryWaves / kWaves);
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x % (kLibraryWaves / kWaves) * kWaves +
                                                    threadIdx.x / TK_WAVE);
    const int lane = threadIdx.x & (TK_WAVE - 1);
    const int total = B * P;
    int at = (wave * TK_WAVE + lane) * V;   // in the channel's values, all rows behind one another
    int column = at;                        // in its row (at < STEP <= P: a step is one row on at most)
    int64_t offset = (int64_t)c * P + at;   // in y
    const int64_t next_row = (int64_t)(C - 1) * P;
    float sum = 0.0f, squares = 0.0f;
    while (at < total) {  // (steps beyond the end read the channel's first values and leave them out)
        vec v[kAhead];
        int left = 0;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const bool there = at < total;
            v[i] = *reinterpret_cast<const vec *>(y + (there ? offset : (int64_t)c * P));
            left += there ? 1 : 0;
            at += STEP;
            column += STEP;
            offset += STEP;
            if (column >= P) {
                column -= P;
                offset += next_row;
            }
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (i < left) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    const float x = V == 1 ? v[i][0] : v[i][j];
                    sum = sum + x;
                    squares = __builtin_fmaf(x, x, squares);
                }
            }
        }
    }
#pragma unroll
    for (int o = 1; o < TK_WAVE; o <<= 1) {
        sum = sum + __shfl_xor(sum, o);
        squares = squares + __shfl_xor(squares, o);
    }
    if (lane == 0)
        partial[c * kLibraryWaves + wave] = make_float2(sum, squares);
}

// The channel's constants from its sixteen sums, left in memory by whoever is `first`.
__device__ __forceinline__ f32x4 batch_constants(const tk3d_mlp_batch_norm &n, int c, bool first)
{
    const float2 *p = reinterpret_cast<const float2 *>(n.partial) + c * kLibraryWaves;
    float sum = p[0].x, squares = p[0].y;
#pragma unroll
    for (int w = 1; w < kLibraryWaves; ++w) {
        sum = sum + p[w].x;
        squares = squares + p[w].y;
    }
    const double total = (double)n.B * n.P;
    const float share = 1.0f / (float)total;
    const float mean = sum * share;
    float variance = __builtin_fmaf(-mean, mean, squares * share);
    variance = variance < 0.0f ? 0.0f : variance;  // (NaN stays)
    const float inv_std = (float)(1.0 / __builtin_sqrt((double)variance + n.eps));
    if (first) {
        n.mean[c] = mean;
        n.inv_std[c] = inv_std;
        const float m = n.momentum, old = n.running_mean[c];
        n.running_mean[c] = __builtin_fmaf(m, mean, __builtin_fmaf(-m, old, old));
        const float unbiased = variance * (float)(total / (total - 1.0));
        n.running_var[c] = __builtin_fmaf(1.0f - m, n.running_var[c], m * unbiased);
    }
    return f32x4{mean, inv_std, n.gamma[c], n.beta[c]};
}

// The batch norm's count of batches, where the caller has one. (A launch of its own for the layers of a chain took 3
// to 4 us.)
__device__ __forceinline__ void count_batch(int64_t *count)
{
    if (count && blockIdx.x == 0 && threadIdx.x == 0)
        *count += 1;
}

// z = relu(norm(y)), a stretch of a row per workgroup.
__global__ void __launch_bounds__(kBlock) batch_relu_kernel(const float *__restrict__ y,
                                                            tk3d_mlp_batch_norm n, int64_t *count,
                                                            float *__restrict__ z, int stretches)
{
    count_batch(count);
    const int part = blockIdx.x % stretches, row = blockIdx.x / stretches, c = row % n.C;
    const f32x4 k = batch_constants(n, c, row < n.C && part == 0 && threadIdx.x == 0);
    const int64_t base = (int64_t)row * n.P;
    const int step = stretches * kBlock * 4;
    int i = (part * kBlock + threadIdx.x) * 4;
    for (; i + 3 * step < n.P; i += 4 * step) {
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = *reinterpret_cast<const f32x4 *>(y + base + i + u * step);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[u][j] = relu(normalised(v[u][j], k));
            *reinterpret_cast<f32x4 *>(z + base + i + u * step) = v[u];
        }
    }
    for (; i < n.P; i += step) {
        f32x4 v = *reinterpret_cast<const f32x4 *>(y + base + i);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = relu(normalised(v[j], k));
        *reinterpret_cast<f32x4 *>(z + base + i) = v;
    }
}

// Largest value of a group of LANES neighbouring lanes, in all of them; NaN above all.
template <int LANES> __device__ __forceinline__ float group_maximum(float v)
{
#define TK_MAXIMUM_STEP(ctrl)                                                                         \
    v = __builtin_elementwise_maximum(                                                                \
        v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true)));
    TK_MAXIMUM_STEP(0xb1)  // quad_perm 1,0,3,2
    TK_MAXIMUM_STEP(0x4e)  // quad_perm 2,3,0,1
    TK_MAXIMUM_STEP(0x141)  // row_half_mirror
    if constexpr (LANES > 8)
        TK_MAXIMUM_STEP(0x140)  // row_mirror
#undef TK_MAXIMUM_STEP
    return v;
}
template <int LANES> __device__ __forceinline__ int group_first(int v)
{
#define TK_FIRST_STEP(ctrl)                                                                           \
    {                                                                                                 \
        const int o = __builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, true);                        \
        v = o < v ? o : v;                                                                            \
    }
    TK_FIRST_STEP(0xb1)
    TK_FIRST_STEP(0x4e)
    TK_FIRST_STEP(0x141)
    if constexpr (LANES > 8)
        TK_FIRST_STEP(0x140)
#undef TK_FIRST_STEP
    return v;
}

// out = relu(max norm(y)) over groups of `size` values, where the maximum is and the y there, the first of
// equals, NaN above all. LANES lanes share a group of 4 LANES values; 0: a lane walks a group.
// The largest value first, then the first place that holds it: three instructions a value beside the
// norm, where a maximum that carries its place and its y along takes nine, and three exchanges through LDS
// a step between lanes. Bound by memory (and the last-level cache) now: [16, 64, 512, 32] 18.2 -> 15.5 us, [16, 128, 512, 32]
// 29.9 -> 24.3, [16, 256, 128, 64] 31.8 -> 24.0. (Over groups of 20, a lane a group, it made no difference.)
template <int LANES>
__global__ void __launch_bounds__(kBlock) batch_pool_kernel(const float *__restrict__ y,
                                                            tk3d_mlp_batch_norm n, int size,
                                                            float *__restrict__ out,
                                                            float *__restrict__ extreme,
                                                            unsigned char *__restrict__ arg,
                                                            int stretches, int64_t *count)
{
    count_batch(count);
    constexpr int NONE = 0x7fffffff;
    const int part = blockIdx.x % stretches, row = blockIdx.x / stretches, c = row % n.C;
    const f32x4 k = batch_constants(n, c, row < n.C && part == 0 && threadIdx.x == 0);
    const int M = n.P / size;
    const float *__restrict__ values = y + (int64_t)row * n.P;
    const int64_t to = (int64_t)row * M;
    const auto put = [&](int g, float z, float raw, int where) {
        out[to + g] = relu(z);
        extreme[to + g] = raw;
        arg[to + g] = (unsigned char)where;
    };
    if constexpr (LANES != 0) {
        constexpr int U = 4;  // groups at once
        const int l = threadIdx.x % LANES, step = stretches * (kBlock / LANES);
        for (int g0 = part * (kBlock / LANES) + threadIdx.x / LANES; g0 < M; g0 += U * step) {
            f32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int g = g0 + u * step < M ? g0 + u * step : g0;
                v[u] = *reinterpret_cast<const f32x4 *>(values + ((int64_t)g * LANES + l) * 4);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                f32x4 z;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    z[i] = normalised(v[u][i], k);
                const float best = group_maximum<LANES>(__builtin_elementwise_maximum(
                    __builtin_elementwise_maximum(z[0], z[1]), __builtin_elementwise_maximum(z[2], z[3])));
                // (nothing is above `best`, and a NaN is where it is one)
                const bool nan = best != best;
                int own = NONE;
                float raw = 0.0f;
#pragma unroll
                for (int i = 3; i >= 0; --i) {
                    const bool here = nan ? z[i] != z[i] : z[i] == best;
                    own = here ? 4 * l + i : own;
                    raw = here ? v[u][i] : raw;
                }
                const int where = group_first<LANES>(own);
                if (own == where && g0 + u * step < M)  // (one lane of the group has it)
                    put(g0 + u * step, best, raw, where);
            }
        }
    } else {
        for (int g = part * kBlock + threadIdx.x; g < M; g += stretches * kBlock) {
            const float *__restrict__ group = values + (int64_t)g * size;
            float raw = group[0], best = normalised(raw, k);
            int where = 0;
            const auto look = [&](float x, int i) {
                const int before = where;
                take_larger(best, where, normalised(x, k), i);
                raw = where != before ? x : raw;
            };
            if ((size & 3) == 0) {
                for (int i = 0; i < size; i += 20) {  // (five loads ahead)
                    f32x4 v[5];
#pragma unroll
                    for (int u = 0; u < 5; ++u)
                        v[u] = *reinterpret_cast<const f32x4 *>(group + (i + 4 * u < size ? i + 4 * u : i));
#pragma unroll
                    for (int u = 0; u < 5; ++u) {
                        if (i + 4 * u < size) {
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (i + 4 * u + j > 0)
                                    look(v[u][j], i + 4 * u + j);
                        }
                    }
                }
            } else {
                for (int i = 1; i < size; ++i)
                    look(group[i], i);
            }
            put(g, best, raw, where);
        }
    }
}

// The same over whole rows, a wave a row; Z: from the normalised values z.
template <bool Z>
__global__ void __launch_bounds__(kBlock)
    batch_rows_kernel(const float *__restrict__ y, const float *__restrict__ z, tk3d_mlp_batch_norm n, int rows, int C,
                      int P, float *__restrict__ out, float *__restrict__ extreme, int *__restrict__ arg,
                      int64_t *__restrict__ index, int64_t *count)
{
    count_batch(count);
    const int row = blockIdx.x * kWaves + threadIdx.x / TK_WAVE, lane = threadIdx.x % TK_WAVE;
    if (row >= rows)
        return;
    f32x4 k{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (!Z)
        k = batch_constants(n, row % C, row < C && lane == 0);
    const float *__restrict__ values = (Z ? z : y) + (int64_t)row * P;
    float best = -__builtin_huge_valf();
    int where = 0x7fffffff;  // (of no value: any other is before it)
    const auto look = [&](float v, int at) { take_larger(best, where, Z ? v : normalised(v, k), at); };
    if ((P & 3) == 0) {
        constexpr int U = 4;
        for (int i = 4 * lane; i < P; i += U * 4 * TK_WAVE) {
            f32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int at = i + u * 4 * TK_WAVE;
                v[u] = *reinterpret_cast<const f32x4 *>(values + (at < P ? at : i));
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i + u * 4 * TK_WAVE < P)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        look(v[u][j], i + u * 4 * TK_WAVE + j);
        }
    } else {
        for (int i = lane; i < P; i += TK_WAVE)
            look(values[i], i);
    }
#pragma unroll
    for (int off = 1; off < TK_WAVE; off <<= 1) {
        const float other = __shfl_xor(best, off);
        const int at = __shfl_xor(where, off);
        take_larger(best, where, other, at);
    }
    if (lane == 0) {
        out[row] = relu(best);
        extreme[row] = y[(int64_t)row * P + where];
        arg[row] = where;
        index[row] = best <= 0.0f ? 0 : where;  // (behind the ReLU all are zero then)
    }
}

// Workgroups per row, so that the chip has sixteen per CU of them and none has under 4096 values.
int stretches_of(int64_t rows, int P)
{
    const int64_t wanted = (16 * (int64_t)tk_cu_count() + rows - 1) / rows, most = (P + 4095) / 4096;
    const int64_t n = wanted < most ? wanted : most;
    return n < 1 ? 1 : (int)n;
}

}  // namespace

extern "C" {

int tk3d_mlp_batch_norm_supported(int64_t B, int64_t C, int64_t P)
{
    // (what has been compared with the library's results; it takes other kernels for rows of up to 1024
    // values, from 2^25 values a channel on and for batches of thousands)
    return B >= 1 && B <= 512 && C >= 1 && C <= 2048 && P > 1024 && P % 4 == 0 && B * P <= (1 << 21);
}

int64_t tk3d_mlp_batch_norm_partial_bytes(int64_t C)
{
    return C * kLibraryWaves * (int64_t)sizeof(float2);
}

int tk3d_mlp_batch_sums_f32(const float *y, int B, int C, int P, void *partial, void *stream)
{
    if (!tk3d_mlp_batch_norm_supported(B, C, P))
        return TK3D_ERR_UNSUPPORTED;
    const bool wide = P >= 4096;
    if (wide && ((uintptr_t)y & 15) != 0)
        return TK3D_ERR_UNSUPPORTED;
    const unsigned grid = (unsigned)(C * (kLibraryWaves / kWaves));
    if (wide)
        batch_sums_kernel<4><<<grid, kBlock, 0, (hipStream_t)stream>>>(
            y, B, C, P, reinterpret_cast<float2 *>(partial));
    else
        batch_sums_kernel<1><<<grid, kBlock, 0, (hipStream_t)stream>>>(
            y, B, C, P, reinterpret_cast<float2 *>(partial));
    return tk_launch_status();
}

int tk3d_mlp_batch_relu_f32(const float *y, const tk3d_mlp_batch_norm *norm, float *z, void *stream)
{
    return tk3d_mlp_batch_relu_counted_f32(y, norm, nullptr, z, stream);
}

int tk3d_mlp_batch_relu_counted_f32(const float *y, const tk3d_mlp_batch_norm *norm, int64_t *count, float *z,
                                    void *stream)
{
    if (!tk3d_mlp_batch_norm_supported(norm->B, norm->C, norm->P) ||
        (((uintptr_t)y | (uintptr_t)z) & 15) != 0)
        return TK3D_ERR_UNSUPPORTED;
    const int64_t rows = (int64_t)norm->B * norm->C;
    const int stretches = stretches_of(rows, norm->P);
    batch_relu_kernel<<<(unsigned)(rows * stretches), kBlock, 0, (hipStream_t)stream>>>(
        y, *norm, count, z, stretches);
    return tk_launch_status();
}

int tk3d_mlp_batch_pool_f32(const float *y, const tk3d_mlp_batch_norm *norm, int size, float *out,
                            float *extreme, unsigned char *arg, void *stream)
{
    return tk3d_mlp_batch_pool_counted_f32(y, norm, nullptr, size, out, extreme, arg, stream);
}

int tk3d_mlp_batch_pool_counted_f32(const float *y, const tk3d_mlp_batch_norm *norm, int64_t *count, int size,
                                    float *out, float *extreme, unsigned char *arg, void *stream_)
{
    if (!tk3d_mlp_batch_norm_supported(norm->B, norm->C, norm->P) || ((uintptr_t)y & 15) != 0)
        return TK3D_ERR_UNSUPPORTED;
    if (size <= 0 || size > 255 || norm->P % size != 0)
        return TK3D_ERR_BAD_SIZE;
    const int64_t rows = (int64_t)norm->B * norm->C;
    const int stretches = stretches_of(rows, norm->P);
    const unsigned grid = (unsigned)(rows * stretches);
    const hipStream_t stream = (hipStream_t)stream_;
    if (size == 32)
        batch_pool_kernel<8><<<grid, kBlock, 0, stream>>>(y, *norm, size, out, extreme, arg, stretches, count);
    else if (size == 64)
        batch_pool_kernel<16><<<grid, kBlock, 0, stream>>>(y, *norm, size, out, extreme, arg, stretches, count);
    else
        batch_pool_kernel<0><<<grid, kBlock, 0, stream>>>(y, *norm, size, out, extreme, arg, stretches, count);
    return tk_launch_status();
}

int tk3d_mlp_batch_rows_f32(const float *y, const float *z, const tk3d_mlp_batch_norm *norm, int B, int C, int P,
                            float *out, float *extreme, int32_t *arg, int64_t *index, void *stream)
{
    return tk3d_mlp_batch_rows_counted_f32(y, z, norm, nullptr, B, C, P, out, extreme, arg, index, stream);
}

int tk3d_mlp_batch_rows_counted_f32(const float *y, const float *z, const tk3d_mlp_batch_norm *norm, int64_t *count,
                                    int B, int C, int P, float *out, float *extreme, int32_t *arg, int64_t *index,
                                    void *stream_)
{
    if (B <= 0 || C <= 0 || P <= 0)
        return TK3D_ERR_BAD_SIZE;
    if (!tk_fits(TK_MAX_I32, B, C) || (P % 4 == 0 && (((uintptr_t)y | (uintptr_t)z) & 15) != 0))
        return TK3D_ERR_UNSUPPORTED;
    const int rows = B * C;
    const unsigned grid = (unsigned)((rows + kWaves - 1) / kWaves);
    const hipStream_t stream = (hipStream_t)stream_;
    if (z)
        batch_rows_kernel<true><<<grid, kBlock, 0, stream>>>(y, z, tk3d_mlp_batch_norm{}, rows, C, P, out, extreme, arg,
                                                            index, count);
    else if (tk3d_mlp_batch_norm_supported(norm->B, norm->C, norm->P))
        batch_rows_kernel<false><<<grid, kBlock, 0, stream>>>(y, z, *norm, rows, C, P, out, extreme, arg, index,
                                                             count);
    else
        return TK3D_ERR_UNSUPPORTED;
    return tk_launch_status();
}

}  // extern "C"
