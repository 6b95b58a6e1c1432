// EdgeConv with one layer, pooled over the neighbours (include/tk3d_mlp.h): the layer is linear in
// the edge feature [x_j - x_i, x_i], so y(i, j) = u_j + v_i with u = W1 x and v = (W2 - W1) x, two
// products per POINT instead of one per edge, and nothing of the size of the edges is ever stored:
// the forward gathers the u of a point's neighbours and keeps the extreme, its place, the sum and
// the statistics; the backward gathers, through the inverse of the graph, what the edges into a
// point contribute. Bound by the L2: a row of 64 channels (256 bytes) per edge and direction.
#include "mlp_common.h"

namespace {

constexpr int kPoints = 32;    // points of a workgroup
constexpr int kChannels = 64;  // channels of a workgroup: a lane is a channel
constexpr int kAtOnce = 8;     // rows requested before the first is used

// out [2 O][C]: W1, then W2 - W1, from w [O][2 C].
__global__ void __launch_bounds__(kBlock) edge_weights_kernel(const float *w, int O, int C, float *out)
{
    const int n = O * C;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const int o = i / C, c = i - o * C;
        const float w1 = w[(int64_t)o * 2 * C + c], w2 = w[(int64_t)o * 2 * C + C + c];
        out[i] = w1;
        out[n + i] = w2 - w1;
    }
}

// A workgroup takes 32 points, a wave eight of them, a lane one of 64 channels. Consecutive
// workgroups take different batch elements, so that an XCD's L2 holds the rows of few.
__global__ void __launch_bounds__(kBlock)
    edge_forward_kernel(const float *__restrict__ uv, const int64_t *__restrict__ index,
                        const float *__restrict__ gamma, int B, int N, int K, int O, int total,
                        float *__restrict__ extreme, float *__restrict__ sum)
{
    __shared__ float values[kChannels][kPoints + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cbase = blockIdx.y * kChannels;
    const int c = cbase + lane < O ? cbase + lane : O - 1;
    const float sign = sign_of(gamma[c]);
    for (int tile = blockIdx.x; tile < total; tile += gridDim.x) {
        const int b = tile % B, first = tile / B * kPoints;
        const float *u = uv + (int64_t)b * N * 2 * O + c;
        for (int q = 0; q < kPoints / kWaves; ++q) {
            const int local = wave * (kPoints / kWaves) + q, i = first + local;
            if (i >= N)
                break;
            const int64_t *row = index + ((int64_t)b * N + i) * K;
            const float v = u[(int64_t)i * 2 * O + O];
            float best = 0.0f, chosen = 0.0f, total_u = 0.0f;
            for (int k0 = 0; k0 < K; k0 += kAtOnce) {
                float r[kAtOnce];
#pragma unroll
                for (int k = 0; k < kAtOnce; ++k) {
                    const int64_t j = row[k0 + k < K ? k0 + k : K - 1];
                    r[k] = j >= 0 && j < N ? u[j * 2 * O] : 0.0f;
                }
#pragma unroll
                for (int k = 0; k < kAtOnce; ++k) {
                    if (k0 + k >= K)
                        break;
                    const float y = r[k] + v;
                    total_u += r[k];
                    const float s = y * sign;
                    // (the first NaN stays, as in torch's maximum)
                    const bool up = k0 + k == 0 || (!(s <= best) && best == best);
                    best = up ? s : best;
                    chosen = up ? y : chosen;
                }
            }
            values[lane][local] = chosen;
            if (sum && cbase + lane < O)
                sum[((int64_t)b * N + i) * O + c] = total_u;
        }
        if (!extreme)
            continue;
        __syncthreads();
        for (int e = tid; e < kChannels * kPoints; e += kBlock) {
            const int ch = e / kPoints, p = e % kPoints;
            if (cbase + ch < O && first + p < N) {
                const int64_t at = ((int64_t)b * O + cbase + ch) * N + first + p;
                extreme[at] = values[ch][p];
            }
        }
        __syncthreads();
    }
}

// The edge features themselves, [x_j - x_i, x_i] as [B, 2 C, N, K] (x_j = 0 for an index outside):
// written once, where group, difference and concatenation were three passes over them and more.
// A thread has four consecutive edges (one where their number is odd) of kEdgeChannels channels.
constexpr int kEdgeChannels = 8;

template <int RUN>
__global__ void __launch_bounds__(kBlock)
    edge_features_kernel(const float *__restrict__ x, const int64_t *__restrict__ index, int C, int N,
                         int K, float *__restrict__ out)
{
    const int b = blockIdx.z, edges = N * K;
    const int cbase = blockIdx.y * kEdgeChannels;
    const int e = (blockIdx.x * kBlock + threadIdx.x) * RUN;
    if (e >= edges)
        return;
    int i[RUN], j[RUN];
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
        const int64_t at = index[(int64_t)b * edges + e + r];
        i[r] = (e + r) / K;
        j[r] = at >= 0 && at < N ? (int)at : -1;
    }
    float *diff = out + (int64_t)b * 2 * C * edges + e, *own = diff + (int64_t)C * edges;
    const float *row = x + (int64_t)b * C * N;
    for (int c = cbase; c < C && c < cbase + kEdgeChannels; ++c) {
        float d[RUN], q[RUN];
#pragma unroll
        for (int r = 0; r < RUN; ++r) {
            q[r] = row[(int64_t)c * N + i[r]];
            d[r] = (j[r] >= 0 ? row[(int64_t)c * N + j[r]] : 0.0f) - q[r];
        }
        if constexpr (RUN == 4) {
            *reinterpret_cast<f32x4 *>(diff + (int64_t)c * edges) = f32x4{d[0], d[1], d[2], d[3]};
            *reinterpret_cast<f32x4 *>(own + (int64_t)c * edges) = f32x4{q[0], q[1], q[2], q[3]};
        } else {
            diff[(int64_t)c * edges] = d[0];
            own[(int64_t)c * edges] = q[0];
        }
    }
}

// The inverse of the graph, one workgroup per batch element: start [N + 1], then the edges into
// every point as i << 8 | k. (Their order within a point is arbitrary; the backward adds them up in
// double.)
__global__ void __launch_bounds__(1024)
    edge_lists_kernel(const int64_t *index, int N, int K, int *lists)
{
    extern __shared__ int cursor[];  // [N]
    __shared__ int waves[16];
    const int tid = threadIdx.x, edges = N * K;
    const int64_t *row = index + (int64_t)blockIdx.x * edges;
    int *start = lists + (int64_t)blockIdx.x * (N + 1 + edges);
    int *entries = start + N + 1;
    for (int j = tid; j < N; j += 1024)
        cursor[j] = 0;
    __syncthreads();
    for (int e = tid; e < edges; e += 1024) {
        const int64_t j = row[e];
        if (j >= 0 && j < N)
            atomicAdd(&cursor[(int)j], 1);
    }
    __syncthreads();
    // exclusive prefix sums: a run of points per thread, then over the threads
    const int run = (N + 1023) / 1024, from = tid * run < N ? tid * run : N;
    const int to = from + run < N ? from + run : N;
    int mine = 0;
    for (int j = from; j < to; ++j)
        mine += cursor[j];
    int scan = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int other = __shfl_up(scan, off);
        scan += (tid & 63) >= off ? other : 0;
    }
    if ((tid & 63) == 63)
        waves[tid >> 6] = scan;
    __syncthreads();
    int base = scan - mine;
    for (int w = 0; w < (tid >> 6); ++w)
        base += waves[w];
    for (int j = from; j < to; ++j) {
        const int count = cursor[j];
        cursor[j] = base;
        start[j] = base;
        base += count;
    }
    if (tid == 1023)
        start[N] = base;
    __syncthreads();
    for (int e = tid; e < edges; e += 1024) {
        const int64_t j = row[e];
        if (j >= 0 && j < N)
            entries[atomicAdd(&cursor[(int)j], 1)] = (e / K) << 8 | (e % K);
    }
}

// The sparse gradient, [B, N, O] of (a e, place), from g, extreme and arg [B, O, N].
__global__ void __launch_bounds__(kBlock)
    edge_select_kernel(const float *g, const float *extreme, const unsigned char *arg, int N, int O,
                       tk3d_mlp_norm norm, const float *coef, int2 *sel)
{
    __shared__ int2 tile[kPoints][kChannels + 1];
    const int tid = threadIdx.x, b = blockIdx.z, first = blockIdx.x * kPoints;
    const int cbase = blockIdx.y * kChannels;
    for (int e = tid; e < kChannels * kPoints; e += kBlock) {
        const int ch = e / kPoints, p = e % kPoints, c = cbase + ch;
        if (c < O && first + p < N) {
            const int64_t at = ((int64_t)b * O + c) * N + first + p;
            const f32x4 ss = constants_of(norm, c);
            const float ev = passes(normalised(extreme[at], ss)) ? g[at] : 0.0f;
            tile[p][ch] = int2{__float_as_int(coef[c * 4] * ev), (int)arg[at]};
        }
    }
    __syncthreads();
    for (int e = tid; e < kChannels * kPoints; e += kBlock) {
        const int p = e / kChannels, ch = e % kChannels;
        if (cbase + ch < O && first + p < N)
            sel[((int64_t)b * N + first + p) * O + cbase + ch] = tile[p][ch];
    }
}

// dy(i, k) = (a e)_i [k is the place] + b y + d, summed over the edges into a point (du) and out of
// it (dv); out [B, 2 O, N]: du, then dv.
__global__ void __launch_bounds__(kBlock)
    edge_backward_kernel(const float *__restrict__ uv, const int2 *__restrict__ sel,
                         const float *__restrict__ sum, const int *__restrict__ lists,
                         const float *__restrict__ coef, int B, int N, int K, int O,
                         float *__restrict__ out)
{
    __shared__ float du[kChannels][kPoints + 1], dv[kChannels][kPoints + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cbase = blockIdx.y * kChannels;
    const int c = cbase + lane < O ? cbase + lane : O - 1;
    const int b = blockIdx.x % B, first = blockIdx.x / B * kPoints;
    const float kb = coef[c * 4 + 1], kd = coef[c * 4 + 2];
    const float *u = uv + (int64_t)b * N * 2 * O + c;
    const int2 *selected = sel + (int64_t)b * N * O + c;
    const int *start = lists + (int64_t)b * (N + 1 + (int64_t)N * K);
    const int *entries = start + N + 1;
    for (int q = 0; q < kPoints / kWaves; ++q) {
        const int local = wave * (kPoints / kWaves) + q, j = first + local;
        if (j >= N)
            break;
        // (the lists come from the caller: whatever they hold, nothing outside is read)
        const int from = min(max(start[j], 0), N * K), to = min(max(start[j + 1], from), N * K);
        double acc = 0.0;
        for (int e0 = from; e0 < to; e0 += kAtOnce) {
            float v[kAtOnce];
            int2 s[kAtOnce];
            int k[kAtOnce];
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) {
                const int entry = entries[e0 + i < to ? e0 + i : to - 1];
                const int64_t at = min((unsigned)entry >> 8, (unsigned)N - 1u);
                k[i] = entry & 255;
                v[i] = u[at * 2 * O + O];
                s[i] = selected[at * O];
            }
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) {
                if (e0 + i >= to)
                    break;
                acc += (double)__builtin_fmaf(kb, v[i], s[i].y == k[i] ? __int_as_float(s[i].x) : 0.0f);
            }
        }
        const float deg = (float)(to - from), all = (float)K;
        const float uj = u[(int64_t)j * 2 * O], vj = u[(int64_t)j * 2 * O + O];
        du[lane][local] = (float)(acc + (double)deg * ((double)kb * (double)uj + (double)kd));
        const float s = sum[((int64_t)b * N + j) * O + c];
        dv[lane][local] = __int_as_float(selected[(int64_t)j * O].x) +
                          __builtin_fmaf(kb, __builtin_fmaf(all, vj, s), all * kd);
    }
    __syncthreads();
    for (int e = tid; e < kChannels * kPoints; e += kBlock) {
        const int ch = e / kPoints, p = e % kPoints;
        if (cbase + ch < O && first + p < N) {
            float *row = out + ((int64_t)b * 2 * O + cbase + ch) * N + first + p;
            row[0] = du[ch][p];
            row[(int64_t)O * N] = dv[ch][p];
        }
    }
}

}  // namespace

extern "C" {

int tk3d_mlp_edge_supported(int64_t B, int64_t N, int64_t K, int64_t O)
{
    return B > 0 && B <= 65535 && N > 0 && N <= 32768 && K > 0 && K <= 255 && O > 0 && O <= 4096 &&
           tk_fits(TK_MAX_I32, B, (N + kPoints - 1) / kPoints) && tk_fits(TK_MAX_I32 / 2, N, K);
}

int tk3d_mlp_edge_weights_f32(const float *w, int O, int C, float *out, void *stream)
{
    const int blocks = (O * C + kBlock - 1) / kBlock;
    edge_weights_kernel<<<blocks < 256 ? blocks : 256, kBlock, 0, (hipStream_t)stream>>>(w, O, C, out);
    return tk_launch_status();
}

int tk3d_mlp_edge_features_f32(const float *x, const int64_t *index, int B, int C, int N, int K,
                               float *out, void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, 1) || C <= 0 || C > 4096)
        return TK3D_ERR_UNSUPPORTED;
    const int edges = N * K, run = edges % 4 == 0 ? 4 : 1;
    const dim3 grid((edges / run + kBlock - 1) / kBlock, (C + kEdgeChannels - 1) / kEdgeChannels, B);
    if (run == 4)
        edge_features_kernel<4><<<grid, kBlock, 0, (hipStream_t)stream>>>(x, index, C, N, K, out);
    else
        edge_features_kernel<1><<<grid, kBlock, 0, (hipStream_t)stream>>>(x, index, C, N, K, out);
    return tk_launch_status();
}

int tk3d_mlp_edge_forward_f32(const float *uv, const int64_t *index, const float *gamma, int B, int N,
                              int K, int O, float *extreme, float *sum, void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, O))
        return TK3D_ERR_UNSUPPORTED;
    const int tiles = B * ((N + kPoints - 1) / kPoints);
    const int most = 4 * tk_cu_count() / B * B;  // (whole rounds of the batch)
    const int blocks = tiles < most || most == 0 ? tiles : most;
    edge_forward_kernel<<<dim3(blocks, (O + kChannels - 1) / kChannels), kBlock, 0, (hipStream_t)stream>>>(
        uv, index, gamma, B, N, K, O, tiles, extreme, sum);
    return tk_launch_status();
}

int tk3d_mlp_edge_lists(const int64_t *index, int B, int N, int K, int32_t *lists, void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, 1))
        return TK3D_ERR_UNSUPPORTED;
    const int rc = tk_allow_dynamic_lds<edge_lists_kernel>(32768 * 4);
    if (rc != TK3D_OK)
        return rc;
    edge_lists_kernel<<<B, 1024, N * 4, (hipStream_t)stream>>>(index, N, K, lists);
    return tk_launch_status();
}

int tk3d_mlp_edge_backward_f32(const float *g, const float *extreme, const unsigned char *arg,
                               const float *uv, const float *sum, const int32_t *lists, int B, int N,
                               int K, int O, const tk3d_mlp_norm *norm, const float *coef, void *sel,
                               float *duv, void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, O))
        return TK3D_ERR_UNSUPPORTED;
    const int tiles = (N + kPoints - 1) / kPoints, blocks = (O + kChannels - 1) / kChannels;
    edge_select_kernel<<<dim3(tiles, blocks, B), kBlock, 0, (hipStream_t)stream>>>(
        g, extreme, arg, N, O, *norm, coef, reinterpret_cast<int2 *>(sel));
    edge_backward_kernel<<<dim3(tiles * B, blocks), kBlock, 0, (hipStream_t)stream>>>(
        uv, reinterpret_cast<const int2 *>(sel), sum, lists, coef, B, N, K, O, duv);
    return tk_launch_status();
}

}  // extern "C"
