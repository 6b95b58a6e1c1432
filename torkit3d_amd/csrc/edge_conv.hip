// EdgeConv with one layer, pooled over the neighbours (include/tk3d_mlp.h). The layer is linear in the
// edge feature [x_j - x_i, x_i], so what runs over the edges are gathers of rows per point, and the
// products are per point: nothing of the size of the edges is stored but what the stock modules leave
// in training. Bound by the L2 (a row of 64 channels, 256 bytes, per edge and direction) and, in the
// products, by the rate of the fp64 matrix instructions (79 TFLOP/s).
//
// Why fp64: y taken apart into a term of j and one of i loses what the difference of near
// neighbours keeps. With fp32 products u + v of [W1 x]_j and [(W2 - W1) x]_i is 1.6 to 2.3 times as far
// from float64 as the product with the edge feature, and dW1 = du x^T - dv x^T up to 2.7 times; with
// fp64 products, rounded once, u + v 0.2 to 0.4 times (C = 64; at C = 3 it would be 1.2 to 1.5 times, so
// that below kRounded channels the sum is rounded and not its terms: 0.7 times), dW1 0.2 to 0.3 and dx
// 0.4 to 0.6 times on clouds about the origin. Far from it both forms are as exact as the statistics
// that the library saved. (With u and v in fp64 at any C DGCNN's evaluation is 3 to 4 % slower.)
#include "mlp_common.h"

namespace {

constexpr int kPoints = 32;    // points of a workgroup
constexpr int kChannels = 64;  // channels of a workgroup: a lane is a channel
constexpr int kGather = 16;    // points of a workgroup that gathers in the backward: waves to hide trips
constexpr int kRounded = 16;   // channels from which u and v may be rounded before they are added
constexpr int kAtOnce = 8;     // rows requested before the first is used
constexpr int kOwners = 512;   // lanes of a workgroup that adds what belongs to neighbours in LDS
constexpr int kPart = 2048;    // its points at a time: every wave's run of 64 x kAtOnce within it
constexpr int kOwnersLds = 144 * 1024;

// The extreme of y = u_j + v_i over the neighbours.
// A workgroup takes 32 points, a wave eight of them, a lane one of 64 output channels. Consecutive
// workgroups take different batch elements, so that an XCD's L2 holds the rows of few.
template <typename T>
__global__ void __launch_bounds__(kBlock)
    edge_forward_kernel(const T *__restrict__ uv, const int64_t *__restrict__ index,
                        const float *__restrict__ gamma, int B, int N, int K, int O, int total,
                        float *__restrict__ extreme)
{
    __shared__ float values[kChannels][kPoints + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cbase = blockIdx.y * kChannels;
    const int c = cbase + lane < O ? cbase + lane : O - 1;
    const float sign = sign_of(gamma[c]);
    for (int tile = blockIdx.x; tile < total; tile += gridDim.x) {
        const int b = tile % B, first = tile / B * kPoints;
        const T *u = uv + (int64_t)b * N * 2 * O + c;
        for (int q = 0; q < kPoints / kWaves; ++q) {
            const int local = wave * (kPoints / kWaves) + q, i = first + local;
            if (i >= N)
                break;
            const int64_t *row = index + ((int64_t)b * N + i) * K;
            const T v = u[(int64_t)i * 2 * O + O];
            float best = 0.0f, chosen = 0.0f;
            for (int k0 = 0; k0 < K; k0 += kAtOnce) {
                T r[kAtOnce];
#pragma unroll
                for (int k = 0; k < kAtOnce; ++k) {
                    const int64_t j = row[k0 + k < K ? k0 + k : K - 1];
                    r[k] = j >= 0 && j < N ? u[j * 2 * O] : (T)0;
                }
#pragma unroll
                for (int k = 0; k < kAtOnce; ++k) {
                    if (k0 + k >= K)
                        break;
                    const float y = (float)(r[k] + v), s = y * sign;
                    // (the first NaN stays, as in torch's maximum)
                    const bool up = k0 + k == 0 || (!(s <= best) && best == best);
                    best = up ? s : best;
                    chosen = up ? y : chosen;
                }
            }
            values[lane][local] = chosen;
        }
        __syncthreads();
        for (int e = tid; e < kChannels * kPoints; e += kBlock) {
            const int ch = e / kPoints, p = e % kPoints;
            if (cbase + ch < O && first + p < N)
                extreme[((int64_t)b * O + cbase + ch) * N + first + p] = values[ch][p];
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

// The inverse of the graph: start [N + 1], then the edges into every point as i << 8 | k. (Their order within
// a point is arbitrary; the backward adds them up in double.) A workgroup has `own` points of a batch element and
// looks through all its edges, counting those into lower points on the way; a thread's indices come eight at a
// time. What bounds it are these trips to memory, and the scattered entries, 64 cache lines a store, of which
// one workgroup per batch element had all (8 x 2048 points, 20 neighbours 43 us, now 20).
__global__ void __launch_bounds__(1024)
    edge_lists_kernel(const int64_t *index, int N, int K, int own, int slices, int *lists)
{
    constexpr int AT_ONCE = 8;
    extern __shared__ int cursor[];  // [own]
    __shared__ int waves[16], lower[16];
    const int tid = threadIdx.x, edges = N * K, b = blockIdx.x / slices;
    const int first = blockIdx.x % slices * own, last = min(first + own, N);
    if (first >= N)
        return;
    const int64_t *row = index + (int64_t)b * edges;
    int *start = lists + (int64_t)b * (N + 1 + edges);
    int *entries = start + N + 1;
    for (int j = tid; j < own; j += 1024)
        cursor[j] = 0;
    __syncthreads();
    const auto for_edges = [&](const auto &f) {  // f(edge, point)
        for (int e0 = tid; e0 < edges; e0 += AT_ONCE * 1024) {
            int64_t j[AT_ONCE];
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                j[i] = row[e0 + i * 1024 < edges ? e0 + i * 1024 : e0];
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                if (e0 + i * 1024 < edges && j[i] >= 0 && j[i] < last)
                    f(e0 + i * 1024, (int)j[i]);
        }
    };
    int below = 0;
    for_edges([&](int, int j) {
        if (j >= first)
            atomicAdd(&cursor[j - first], 1);
        else
            ++below;
    });
    __syncthreads();
    // exclusive prefix sums: a run of points per thread, then over the threads; in front of them `below` of all
    const int n = last - first, run = (n + 1023) / 1024, from = tid * run < n ? tid * run : n;
    const int to = from + run < n ? from + run : n;
    int mine = 0;
    for (int j = from; j < to; ++j)
        mine += cursor[j];
    int scan = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int other = __shfl_up(scan, off);
        scan += (tid & 63) >= off ? other : 0;
        below += __shfl_xor(below, off);
    }
    if ((tid & 63) == 63) {
        waves[tid >> 6] = scan;
        lower[tid >> 6] = below;
    }
    __syncthreads();
    int base = scan - mine;
    for (int w = 0; w < 16; ++w)
        base += lower[w] + (w < (tid >> 6) ? waves[w] : 0);
    for (int j = from; j < to; ++j) {
        const int count = cursor[j];
        cursor[j] = base;
        start[first + j] = base;
        base += count;
    }
    if (tid == 1023 && last == N)
        start[N] = base;
    __syncthreads();
    for_edges([&](int e, int j) {
        if (j >= first)
            entries[atomicAdd(&cursor[j - first], 1)] = (e / K) << 8 | (e % K);
    });
}

// The edges into point j, as positions of the entries. (The lists come from the caller: whatever they
// hold, nothing outside is read.)
struct Run {
    int from, to;
};
__device__ __forceinline__ Run edges_into(const int *start, int j, int N, int K)
{
    const int from = min(max(start[j], 0), N * K);
    return {from, min(max(start[j + 1], from), N * K)};
}
__device__ __forceinline__ int point_of(int entry, int N)
{
    return min((unsigned)entry >> 8, (unsigned)N - 1u);
}

// A thread's part of a tile of kChannels by kPoints: a point, and every kChannelStep-th channel. Its loads leave
// together, of the channels that some thread has: one value after the other, each behind the trip of the one before,
// edge_rows_kernel took 6.2 us for 4.8 now (8 x 2048 points, 64 channels), edge_select_kernel 11.2 for 6.3 on those
// sizes, which no longer come to it.
constexpr int kChannelStep = kBlock / kPoints, kOwn = kChannels / kChannelStep;
template <typename F> __device__ __forceinline__ void for_own_channels(int cbase, int channels, const F &load)
{
    if (cbase + kChannels <= channels) {  // uniform, as the others are: a whole tile's loads without them in between
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
            load(i);
    } else {
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
            if (cbase + i * kChannelStep < channels)
                load(i);
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
    const int p = tid % kPoints, ch0 = tid / kPoints;
    float y[kOwn] = {}, gv[kOwn] = {}, a[kOwn] = {};
    int place[kOwn] = {};
    f32x4 ss[kOwn] = {};
    for_own_channels(cbase, O, [&](int i) {  // (what does not exist is read where something else is, and not written)
        const int c = min(cbase + ch0 + i * kChannelStep, O - 1);
        const int64_t at = ((int64_t)b * O + c) * N + min(first + p, N - 1);
        y[i] = extreme[at];
        gv[i] = g[at];
        place[i] = arg[at];
        ss[i] = constants_of(norm, c);
        a[i] = coef[c * 4];
    });
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
        tile[p][ch0 + i * kChannelStep] =
            int2{__float_as_int(a[i] * (passes(normalised(y[i], ss[i])) ? gv[i] : 0.0f)), place[i]};
    __syncthreads();
    for (int e = tid; e < kChannels * kPoints; e += kBlock) {
        const int p = e / kChannels, ch = e % kChannels;
        if (cbase + ch < O && first + p < N)
            sel[((int64_t)b * N + first + p) * O + cbase + ch] = tile[p][ch];
    }
}

// What the sparse gradient adds to du and dv: out [B, 2 O, N], the a e of the edges into a point whose
// place they are, then a point's own.
__global__ void __launch_bounds__(kBlock)
    edge_sparse_kernel(const int2 *__restrict__ sel, const int *__restrict__ lists, int B, int N, int K,
                       int O, float *__restrict__ out)
{
    __shared__ float du[kChannels][kGather + 1], dv[kChannels][kGather + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cbase = blockIdx.y * kChannels;
    const int c = cbase + lane < O ? cbase + lane : O - 1;
    const int b = blockIdx.x % B, first = blockIdx.x / B * kGather;
    const int2 *selected = sel + (int64_t)b * N * O + c;
    const int *start = lists + (int64_t)b * (N + 1 + (int64_t)N * K);
    const int *entries = start + N + 1;
    for (int q = 0; q < kGather / kWaves; ++q) {
        const int local = wave * (kGather / kWaves) + q, j = first + local;
        if (j >= N)
            break;
        const Run run = edges_into(start, j, N, K);
        double acc = 0.0;
        for (int e0 = run.from; e0 < run.to; e0 += kAtOnce) {
            int2 s[kAtOnce];
            int k[kAtOnce];
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) {
                const int entry = entries[e0 + i < run.to ? e0 + i : run.to - 1];
                k[i] = entry & 255;
                s[i] = selected[(int64_t)point_of(entry, N) * O];
            }
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i)
                if (e0 + i < run.to && s[i].y == k[i])
                    acc += (double)__int_as_float(s[i].x);
        }
        du[lane][local] = (float)acc;
        dv[lane][local] = __int_as_float(selected[(int64_t)j * O].x);
    }
    __syncthreads();
    for (int e = tid; e < kChannels * kGather; e += kBlock) {
        const int ch = e / kGather, p = e % kGather;
        if (cbase + ch < O && first + p < N) {
            float *row = out + ((int64_t)b * 2 * O + cbase + ch) * N + first + p;
            row[0] = du[ch][p];
            row[(int64_t)O * N] = dv[ch][p];
        }
    }
}

// The same from g, extreme and arg themselves: a workgroup has CH channels of a cloud, whose sums lie in LDS. kPart
// points at a time, every lane finds the values of its points and the neighbours that they belong to; then one wave a
// channel adds them, 64 points to an atomic. Lanes that meet at a neighbour are taken in their order, so that every
// run adds in that of the points: the hardware's doing, which nothing here enforces and a test holds. The two kernels
// above look at all K edges into a point for the few that count, 8 bytes a channel of each, and pass 8 bytes a value
// through memory; here a value looks up its one neighbour. 8 x 2048 points, 20 neighbours, 64 channels: 26.4 us in
// two launches, now 10.5, most of it the trips to g, to the neighbours and through LDS, one behind the other; 128
// channels 40.8, 14. A step of DGCNN's training on them 74 us less.
template <int CH>
__global__ void __launch_bounds__(kOwners)
    edge_owners_kernel(const float *__restrict__ g, const float *__restrict__ extreme,
                       const unsigned char *__restrict__ arg, const int64_t *__restrict__ index, int B, int N, int K,
                       int O, tk3d_mlp_norm norm, const float *__restrict__ coef, float *__restrict__ out)
{
    extern __shared__ double sums[];  // CH rows of N, then values and neighbours, CH rows of kPart each
    float *values = reinterpret_cast<float *>(sums + CH * N);
    int *owners = reinterpret_cast<int *>(values + CH * kPart);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x % B, c0 = blockIdx.x / B * CH;
    const int64_t *neighbours = index + (int64_t)b * N * K;
    f32x4 ss[CH];
    float a[CH];
    int64_t row[CH];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        const int c = min(c0 + ch, O - 1);
        ss[ch] = constants_of(norm, c);
        a[ch] = coef[c * 4];
        row[ch] = ((int64_t)b * O + c) * N;
    }
    for (int e = tid; e < CH * N; e += kOwners)
        sums[e] = 0.0;
    constexpr int STEPS = kPart / kOwners;
    for (int from = 0; from < N; from += kPart) {
        float y[STEPS][CH], gv[STEPS][CH];
        int place[STEPS][CH];
        int64_t j[STEPS][CH];
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const int p = min(from + i * kOwners + tid, N - 1);
#pragma unroll
            for (int ch = 0; ch < CH; ++ch) {
                place[i][ch] = arg[row[ch] + p];
                y[i][ch] = extreme[row[ch] + p];
                gv[i][ch] = g[row[ch] + p];
            }
        }
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const int p = min(from + i * kOwners + tid, N - 1);
#pragma unroll
            for (int ch = 0; ch < CH; ++ch)
                j[i][ch] = neighbours[(int64_t)p * K + min(place[i][ch], K - 1)];
        }
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const int p = from + i * kOwners + tid;
#pragma unroll
            for (int ch = 0; ch < CH; ++ch) {
                const float v = a[ch] * (passes(normalised(y[i][ch], ss[ch])) ? gv[i][ch] : 0.0f);
                const bool counts = p < N && place[i][ch] < K && j[i][ch] >= 0 && j[i][ch] < N && v != 0.0f;
                values[ch * kPart + i * kOwners + tid] = v;
                owners[ch * kPart + i * kOwners + tid] = counts ? (int)j[i][ch] : -1;
                if (p < N && c0 + ch < O)
                    out[((int64_t)b * 2 * O + O + c0 + ch) * N + p] = v;
            }
        }
        __syncthreads();
        if (wave < CH)
            for (int e0 = 0; e0 < min(kPart, N - from); e0 += 64 * kAtOnce) {
                int to[kAtOnce];
                float v[kAtOnce];
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i) {
                    to[i] = owners[wave * kPart + e0 + i * 64 + lane];
                    v[i] = values[wave * kPart + e0 + i * 64 + lane];
                }
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i)
                    if (to[i] >= 0)
                        unsafeAtomicAdd(&sums[wave * N + to[i]], (double)v[i]);
            }
        __syncthreads();
    }
#pragma unroll
    for (int ch = 0; ch < CH; ++ch)
        if (c0 + ch < O)
            for (int p = tid; p < N; p += kOwners)
                out[((int64_t)b * 2 * O + c0 + ch) * N + p] = (float)sums[ch * N + p];
}

int64_t owners_lds(int N, int channels) { return (int64_t)channels * (N * 8 + kPart * 8); }

// Rows up to here are added in LDS whatever the device; what longer ones take depends on its CUs.
bool may_gather(int N) { return N > 3 * kPart; }

template <int CH>
int edge_owners(const float *g, const float *extreme, const unsigned char *arg, const int64_t *index, int B, int N,
                int K, int O, const tk3d_mlp_norm &norm, const float *coef, float *out, hipStream_t stream)
{
    const int rc = tk_allow_dynamic_lds<edge_owners_kernel<CH>>(kOwnersLds);
    if (rc != TK3D_OK)
        return rc;
    edge_owners_kernel<CH><<<(O + CH - 1) / CH * B, kOwners, owners_lds(N, CH), stream>>>(g, extreme, arg, index, B,
                                                                                         N, K, O, norm, coef, out);
    return tk_launch_status();
}

// x [B, C, N] as rows of points [B, N, C].
__global__ void __launch_bounds__(kBlock) edge_rows_kernel(const float *x, int C, int N, float *rows)
{
    __shared__ float tile[kPoints][kChannels + 1];
    const int tid = threadIdx.x, first = blockIdx.x * kPoints, cbase = blockIdx.y * kChannels;
    const int64_t b = blockIdx.z;
    const int p = tid % kPoints, ch0 = tid / kPoints;
    float v[kOwn] = {};
    for_own_channels(cbase, C, [&](int i) {
        v[i] = x[(b * C + min(cbase + ch0 + i * kChannelStep, C - 1)) * N + min(first + p, N - 1)];
    });
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
        tile[p][ch0 + i * kChannelStep] = v[i];
    __syncthreads();
    for (int e = tid; e < kChannels * kPoints; e += kBlock) {
        const int p = e / kChannels, ch = e % kChannels;
        if (cbase + ch < C && first + p < N)
            rows[(b * N + first + p) * C + cbase + ch] = tile[p][ch];
    }
}

// The edges into a wave's kEach consecutive points, 64 entries of each on their way before the first is used: a lane
// holds an entry, from which its row is read at an address of the whole wave.
constexpr int kEach = kGather / kWaves;
struct Edges {
    Run run[kEach];
    int entry[kEach];
    __device__ __forceinline__ void request(const int *start, const int *entries, int first, int N, int K, int lane)
    {
#pragma unroll
        for (int q = 0; q < kEach; ++q)
            run[q] = edges_into(start, min(first + q, N - 1), N, K);
#pragma unroll
        for (int q = 0; q < kEach; ++q)
            entry[q] = more(entries, q, 0, lane);
    }
    __device__ __forceinline__ int more(const int *entries, int q, int c0, int lane) const
    {
        return run[q].to > run[q].from ? entries[min(run[q].from + c0 + lane, run[q].to - 1)] : 0;
    }
};

// The sums of the differences to the neighbours, out [B, 2 C, N]: s = sum of x_i - x_j over the edges
// i -> j into a point, then t = sum of x_j - x_i over the edges out of it (x_j = 0 outside the cloud).
// W of them lie side by side in a wave: channels of one point. With 64, bounds, edges and neighbours of a wave's points
// are requested at once, and rows of both kinds go together: one behind the other they were twelve trips to memory a
// point (8 x 2048 points, 64 channels, 20 neighbours 34 us, now 24.5; the same for edge_sparse_kernel gave nothing, nor
// did places of a byte there, read in front of the values: 23 -> 26).
template <int W>
__global__ void __launch_bounds__(kBlock)
    edge_neighbours_kernel(const float *__restrict__ rows, const int64_t *__restrict__ index,
                           const int *__restrict__ lists, int B, int N, int K, int C,
                           float *__restrict__ out)
{
    __shared__ float into[W][kGather + 1], from[W][kGather + 1];
    constexpr int AT_ONCE = kBlock / W;  // points
    const int tid = threadIdx.x, lane = tid % W;
    const int sub = W == 64 ? __builtin_amdgcn_readfirstlane(tid / W) : tid / W;
    const int cbase = blockIdx.y * W;
    const int c = cbase + lane < C ? cbase + lane : C - 1;
    const int b = blockIdx.x % B, first = blockIdx.x / B * kGather;
    const float *x = rows + (int64_t)b * N * C + c;
    const int *start = lists + (int64_t)b * (N + 1 + (int64_t)N * K);
    const int *entries = start + N + 1;
    if constexpr (W == 64) {  // (in the same order as below, edges into and out of a point side by side)
        Edges mine;
        mine.request(start, entries, first + sub * kEach, N, K, lane);
        const int64_t *neighbours = index + (int64_t)b * N * K;
        const auto neighbour = [&](int p, int k) {
            const int64_t j = neighbours[(int64_t)min(p, N - 1) * K + min(k, K - 1)];
            return j >= 0 && j < N ? (int)j : -1;
        };
        int out_of[kEach];
        float own[kEach];
#pragma unroll
        for (int q = 0; q < kEach; ++q) {
            out_of[q] = neighbour(first + sub * kEach + q, lane);
            own[q] = x[(int64_t)min(first + sub * kEach + q, N - 1) * C];
        }
#pragma unroll
        for (int q = 0; q < kEach; ++q) {
            const int local = sub * kEach + q, p = first + local;
            if (p >= N)
                break;
            double s = 0.0, t = 0.0;
            const int count = mine.run[q].to - mine.run[q].from;
            for (int c0 = 0; c0 < max(count, K); c0 += 64) {
                const int entry = c0 && c0 < count ? mine.more(entries, q, c0, lane) : mine.entry[q];
                const int near = c0 && c0 < K ? neighbour(p, c0 + lane) : out_of[q];
                const int n = min(count - c0, 64), m = min(K - c0, 64);
                for (int e0 = 0; e0 < max(n, m); e0 += kAtOnce) {
                    float v[kAtOnce], u[kAtOnce];
                    if (e0 < n)
#pragma unroll
                        for (int i = 0; i < kAtOnce; ++i)
                            v[i] = x[(int64_t)point_of(__builtin_amdgcn_readlane(entry, min(e0 + i, n - 1)), N) * C];
                    if (e0 < m)
#pragma unroll
                        for (int i = 0; i < kAtOnce; ++i) {
                            const int j = __builtin_amdgcn_readlane(near, min(e0 + i, m - 1));
                            u[i] = x[(int64_t)max(j, 0) * C];
                            u[i] = j >= 0 ? u[i] : 0.0f;
                        }
                    if (e0 < n)
#pragma unroll
                        for (int i = 0; i < kAtOnce; ++i)
                            s += e0 + i < n ? (double)(v[i] - own[q]) : 0.0;
                    if (e0 < m)
#pragma unroll
                        for (int i = 0; i < kAtOnce; ++i)
                            t += e0 + i < m ? (double)(u[i] - own[q]) : 0.0;
                }
            }
            into[lane][local] = (float)s;
            from[lane][local] = (float)t;
        }
    } else {
        for (int local = sub; local < kGather && first + local < N; local += AT_ONCE) {
            const int p = first + local;
            const float own = x[(int64_t)p * C];
            const Run run = edges_into(start, p, N, K);
            double s = 0.0, t = 0.0;
            for (int e0 = run.from; e0 < run.to; e0 += kAtOnce) {
                float v[kAtOnce];
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i)
                    v[i] = x[(int64_t)point_of(entries[e0 + i < run.to ? e0 + i : run.to - 1], N) * C];
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i)
                    s += e0 + i < run.to ? (double)(v[i] - own) : 0.0;
            }
            const int64_t *neighbours = index + ((int64_t)b * N + p) * K;
            for (int k0 = 0; k0 < K; k0 += kAtOnce) {
                float v[kAtOnce];
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i) {
                    const int64_t j = neighbours[k0 + i < K ? k0 + i : K - 1];
                    v[i] = j >= 0 && j < N ? x[j * C] : 0.0f;
                }
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i)
                    t += k0 + i < K ? (double)(v[i] - own) : 0.0;
            }
            into[lane][local] = (float)s;
            from[lane][local] = (float)t;
        }
    }
    __syncthreads();
    for (int e = tid; e < W * kGather; e += kBlock) {
        const int ch = e / kGather, p = e % kGather;
        if (cbase + ch < C && first + p < N) {
            float *row = out + ((int64_t)b * 2 * C + cbase + ch) * N + first + p;
            row[0] = into[ch][p];
            row[(int64_t)C * N] = from[ch][p];
        }
    }
}

// ---- the products, in fp64 -------------------------------------------------------------------------
//
// result(m, n) = sum over k of a(m, k) b(k, n) for what an Op makes of its tensors: 64 x 64 results a
// workgroup, 32 x 32 a wave (2 x 2 tiles of the 16 x 16 x 4 instruction), sixteen k at a time in LDS,
// the next sixteen requested before these are multiplied. Rows of LDS are 82 doubles: writes along k
// then meet few banks twice. An Op loads what an element is made of (m, n and k clamped to the last)
// and makes it of that in a second function, called when the element goes to LDS: the loads are in
// flight during a whole step. (8 x 2048 points, mean over DGCNN's four blocks: gradients 27 us, weights
// 15, input 16; 44, 29 and 24 where the loading function made the element, and so waited for it.)

typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kTile = 64, kDepth = 16, kPitch = kTile + 18;

struct Raw {
    float p, q;
};
struct Rest {  // of a result: times * sum + plus
    double times, plus;
};

template <typename Op> __global__ void __launch_bounds__(kBlock) edge_product_kernel(Op op)
{
    __shared__ double at[kDepth][kPitch], bt[kDepth][kPitch];
    constexpr int EACH = kTile * kDepth / kBlock;  // elements of either tile a thread loads
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile, z = blockIdx.z;
    const int from = op.from(z), to = op.to(z);
    // (consecutive threads walk the direction in which the tensor lies in memory)
    const auto place = [&](bool along_k, int i, int &k, int &x) {
        k = along_k ? tid % kDepth : tid / kTile + kBlock / kTile * i;
        x = along_k ? tid / kDepth + kBlock / kDepth * i : tid % kTile;
    };
    int am[EACH], bn[EACH];
    double column[EACH];  // what b() wants to know of its n
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        int k, x;
        place(Op::kAlongKA, i, k, x);
        am[i] = min(m0 + x, op.rows - 1);
        place(Op::kAlongKB, i, k, x);
        bn[i] = min(n0 + x, op.cols - 1);
        column[i] = op.column(bn[i], z, m0);
    }
    Raw ar[EACH], br[EACH];
    const auto load = [&](int k0) {
        const int b = op.batch(z, k0);
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
            int k, x;
            place(Op::kAlongKA, i, k, x);
            ar[i] = op.load_a(am[i], op.clamped(min(k0 + k, to - 1), b), b);
            place(Op::kAlongKB, i, k, x);
            br[i] = op.load_b(bn[i], op.clamped(min(k0 + k, to - 1), b), b, m0);
        }
    };
    f64x4 acc[2][2] = {};
    const int row = (wave >> 1) * 32, col = (wave & 1) * 32;
    load(from);
    for (int k0 = from; k0 < to; k0 += kDepth) {
        const int b = op.batch(z, k0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
            int k, x;
            place(Op::kAlongKA, i, k, x);
            const double av = op.a(ar[i], am[i], k0 + k);
            at[k][x] = k0 + k < to && op.inside(k0 + k, b) ? av : 0.0;
            place(Op::kAlongKB, i, k, x);
            const double bv = op.b(br[i], bn[i], k0 + k, column[i]);
            bt[k][x] = k0 + k < to && op.inside(k0 + k, b) ? bv : 0.0;
        }
        __syncthreads();
        if (k0 + kDepth < to)
            load(k0 + kDepth);
#pragma unroll
        for (int k = 0; k < kDepth; k += 4) {
            double a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = at[k + (lane >> 4)][row + 16 * i + (lane & 15)];
                b[i] = bt[k + (lane >> 4)][col + 16 * i + (lane & 15)];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    // (everything that the results are put together with is requested before the first store)
    Rest rest[2][2][4];
    const auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    f(m0 + row + 16 * i + 4 * v + (lane >> 4), n0 + col + 16 * j + (lane & 15),
                      rest[i][j][v], acc[i][j][v]);
    };
    each([&](int m, int n, Rest &r, double) {
        r = op.rest(min(m, op.rows - 1), min(n, op.cols - 1), z);
    });
    each([&](int m, int n, const Rest &r, double sum) {
        if (m < op.rows && n < op.cols)
            op.store(m, n, z, __builtin_fma(r.times, sum, r.plus));
    });
}

// What most Ops have nothing to say about. (The functions a() and b() ignore what they do not need.)
struct PlainOp {
    __device__ int batch(int z, int) const { return z; }
    __device__ int from(int) const { return 0; }
    __device__ int clamped(int k, int) const { return k; }
    __device__ bool inside(int, int) const { return true; }
    __device__ double column(int, int, int) const { return 0.0; }
    __device__ Rest rest(int, int, int) const { return {1.0, 0.0}; }
};

// uv [B, N, 2 O]: a point a row, u = W1 x then v = (W2 - W1) x. m = points, n = u and v, k = channels.
template <typename T> struct EdgeTermsOp : PlainOp {
    static constexpr bool kAlongKA = false, kAlongKB = true;
    const float *x, *w;
    T *uv;
    int C, O, rows, cols;  // rows = N, cols = 2 O
    __device__ int to(int) const { return C; }
    __device__ Raw load_a(int p, int c, int b) const
    {
        return {(x + (int64_t)b * C * rows)[(unsigned)(c * rows + p)], 0.0f};
    }
    __device__ double a(Raw r, int, int) const { return r.p; }
    __device__ Raw load_b(int n, int c, int, int) const
    {
        const unsigned at = (n < O ? n : n - O) * 2 * C + c;
        return {w[at], w[at + C]};
    }
    __device__ double b(Raw r, int n, int, double) const { return n < O ? r.p : (double)r.q - (double)r.p; }
    __device__ void store(int p, int n, int b, double v) const
    {
        uv[((int64_t)b * rows + p) * cols + n] = (T)v;
    }
};

// duv [B, 2 O, N] in place, from the sparse parts: the sum of dy = a e + b (y - mean) + d0 over the
// edges into a point (du) and out of it (dv). y is linear in the edge feature:
//     into j:   sum of y = (W2 - W1) s_j + W2 (deg x_j)
//     out of i: sum of y = W1 t_i + W2 (K x_i)
// m = du then dv, `half` each (a multiple of the tile: a block is all du or all dv), n = points, k =
// the channels of s or t, then those of x.
struct EdgeGradOp : PlainOp {
    static constexpr bool kAlongKA = true, kAlongKB = false;
    const float *x, *st, *w, *coef, *mean;  // st [B, 2 C, N]: s, then t
    const int *lists;
    float *duv;
    int C, O, K, half, rows, cols;  // rows = 2 half, cols = N
    __device__ int to(int) const { return 2 * C; }
    __device__ int edges(int p, int b, bool out) const
    {
        if (out)
            return K;
        const Run run = edges_into(lists + (int64_t)b * (cols + 1 + (int64_t)cols * K), p, cols, K);
        return run.to - run.from;
    }
    __device__ int channel(int m) const { return min(m >= half ? m - half : m, O - 1); }
    __device__ Raw load_a(int m, int k, int) const
    {
        const unsigned row = channel(m) * 2 * C;  // (W1, W2 side by side)
        return {w[row + k], w[row + min(k + C, 2 * C - 1)]};
    }
    __device__ double a(Raw r, int m, int k) const
    {
        return m >= half || k >= C ? r.p : (double)r.q - (double)r.p;
    }
    __device__ double column(int p, int b, int m0) const { return edges(p, b, m0 >= half); }
    __device__ Raw load_b(int p, int k, int b, int m0) const
    {
        const float *own = x + (int64_t)b * C * cols;
        const float *sums = st + ((int64_t)b * 2 + (m0 >= half)) * C * cols;
        return {(k < C ? sums : own)[(unsigned)((k < C ? k : k - C) * cols + p)], 0.0f};
    }
    __device__ double b(Raw r, int, int k, double count) const { return k < C ? r.p : count * (double)r.p; }
    __device__ float *result(int m, int p, int b) const
    {
        return duv + ((int64_t)b * 2 * O + (m >= half ? O : 0) + channel(m)) * cols + p;
    }
    __device__ Rest rest(int m, int p, int b) const
    {
        const f32x4 k = reinterpret_cast<const f32x4 *>(coef)[channel(m)];
        const double n = edges(p, b, m >= half);
        return {k.y, (double)*result(m, p, b) + n * ((double)k.w - (double)k.y * (double)mean[channel(m)])};
    }
    __device__ void store(int m, int p, int b, double v) const
    {
        if ((m >= half ? m - half : m) < O)
            *result(m, p, b) = (float)v;
    }
};

// dx [B, C, N] = W1^T du + (W2 - W1)^T dv. m = channels, n = points, k = du then dv.
struct EdgeInputOp : PlainOp {
    static constexpr bool kAlongKA = false, kAlongKB = false;
    const float *duv, *w;
    float *dx;
    int O, rows, cols;  // rows = C, cols = N
    __device__ int to(int) const { return 2 * O; }
    __device__ Raw load_a(int c, int k, int) const
    {
        const unsigned at = (k < O ? k : k - O) * 2 * rows + c;
        return {w[at], w[at + rows]};
    }
    __device__ double a(Raw r, int, int k) const { return k < O ? r.p : (double)r.q - (double)r.p; }
    __device__ Raw load_b(int p, int k, int b, int) const
    {
        return {(duv + (int64_t)b * 2 * O * cols)[(unsigned)(k * cols + p)], 0.0f};
    }
    __device__ double b(Raw r, int, int, double) const { return r.p; }
    __device__ void store(int c, int p, int b, double v) const
    {
        dx[((int64_t)b * rows + c) * cols + p] = (float)v;
    }
};

// dW1 = (du - dv) x^T and dW2 = dv x^T, partial[z][2 half][C]. The dv of a channel add up to zero, so
// dW2 may count x from its first point: their rounding then does not meet how far x is from zero. (The
// du do so only where no neighbour is outside the cloud.) m = rows of dW1 then of dW2, n = channels, k =
// the points of all batch elements, each filled up to `padded`, a multiple of the depth.
struct EdgeWeightOp : PlainOp {
    static constexpr bool kAlongKA = true, kAlongKB = true;
    const float *x, *duv;
    double *partial;
    int N, O, half, padded, run, total, rows, cols;  // rows = 2 half, cols = C
    __device__ int batch(int, int k0) const { return k0 / padded; }
    __device__ int from(int z) const { return z * run; }
    __device__ int to(int z) const { return total - z * run < run ? total : (z + 1) * run; }
    __device__ int clamped(int k, int b) const { return min(k - b * padded, N - 1); }
    __device__ bool inside(int k, int b) const { return k - b * padded < N; }
    __device__ Raw load_a(int m, int p, int b) const
    {
        const float *du = duv + (int64_t)b * 2 * O * N, *dv = du + (int64_t)O * N;
        const unsigned at = min(m >= half ? m - half : m, O - 1) * N + p;
        return {du[at], dv[at]};
    }
    __device__ double a(Raw r, int m, int) const { return m >= half ? r.q : (double)r.p - (double)r.q; }
    __device__ double column(int c, int, int m0) const { return m0 >= half ? x[(int64_t)c * N] : 0.0f; }
    __device__ Raw load_b(int c, int p, int b, int) const
    {
        return {(x + (int64_t)b * cols * N)[(unsigned)(c * N + p)], 0.0f};
    }
    __device__ double b(Raw r, int, int, double origin) const { return (double)r.p - origin; }
    __device__ void store(int m, int c, int z, double v) const
    {
        partial[((int64_t)z * rows + m) * cols + c] = v;
    }
};

// dw [O][2 C] from the partial sums: sixteen outputs to a workgroup, sixteen threads to an output.
__global__ void __launch_bounds__(kBlock)
    edge_weight_sum_kernel(const double *partial, int parts, int half, int O, int C, float *dw)
{
    __shared__ double lds[kWaves][16];
    const int at = threadIdx.x & 15, lane = threadIdx.x >> 4, i = blockIdx.x * 16 + at;
    const int m = i / C, c = i - m * C, o = m < half ? m : m - half;
    const bool mine = m < 2 * half && o < O;
    double sum = 0.0;
    if (mine)
        for (int z = lane; z < parts; z += 16)
            sum += partial[((int64_t)z * 2 * half + m) * C + c];
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if ((threadIdx.x & 63) < 16)
        lds[threadIdx.x >> 6][at] = sum;
    __syncthreads();
    if (threadIdx.x < 16 && mine)
        dw[(int64_t)o * 2 * C + (m < half ? 0 : C) + c] =
            (float)(lds[0][at] + lds[1][at] + lds[2][at] + lds[3][at]);
}

int tiles_of(int n) { return (n + kTile - 1) / kTile; }

// The points of the weight gradient: padded per batch element, in all, and of one workgroup - four
// workgroups to a CU, and no less than 128 points.
struct WeightRuns {
    int padded, total, run, parts;
};
WeightRuns weight_runs(int B, int N, int O, int C)
{
    WeightRuns r;
    r.padded = (N + kDepth - 1) / kDepth * kDepth;
    r.total = B * r.padded;
    const int blocks = 2 * tiles_of(O) * tiles_of(C), want = (4 * tk_cu_count() + blocks - 1) / blocks;
    r.run = ((r.total + want - 1) / want + kDepth - 1) / kDepth * kDepth;
    r.run = r.run < 128 ? 128 : r.run;
    r.parts = (r.total + r.run - 1) / r.run;
    return r;
}

template <typename Op> int launch_product(const Op &op, int batches, hipStream_t stream)
{
    edge_product_kernel<Op><<<dim3(tiles_of(op.cols), tiles_of(op.rows), batches), kBlock, 0, stream>>>(op);
    return tk_launch_status();
}

template <typename T>
int edge_forward(const float *x, const int64_t *index, const float *w, const float *gamma, int B, int N,
                 int K, int C, int O, T *uv, float *extreme, hipStream_t stream)
{
    const EdgeTermsOp<T> op{{}, x, w, uv, C, O, N, 2 * O};
    const int rc = launch_product(op, B, stream);
    if (rc != TK3D_OK)
        return rc;
    const int tiles = B * ((N + kPoints - 1) / kPoints);
    const int most = 4 * tk_cu_count() / B * B;  // (whole rounds of the batch)
    const dim3 grid(tiles < most || most == 0 ? tiles : most, (O + kChannels - 1) / kChannels);
    edge_forward_kernel<T><<<grid, kBlock, 0, stream>>>(uv, index, gamma, B, N, K, O, tiles, extreme);
    return tk_launch_status();
}

}  // namespace

extern "C" {

int tk3d_mlp_edge_supported(int64_t B, int64_t N, int64_t K, int64_t O)
{
    return B > 0 && B <= 65535 && N > 0 && N <= 32768 && K > 0 && K <= 255 && O > 0 && O <= 4096 &&
           tk_fits(TK_MAX_I32 / 2, B, N + kPoints) && tk_fits(TK_MAX_I32 / 2, N, K);
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

int64_t tk3d_mlp_edge_forward_bytes(int B, int N, int C, int O)
{
    return (int64_t)B * N * 2 * O * (C < kRounded ? 8 : 4);
}

int tk3d_mlp_edge_forward_f32(const float *x, const int64_t *index, const float *w, const float *gamma,
                              int B, int N, int K, int C, int O, void *workspace, float *extreme,
                              void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, O) || C <= 0 || C > 4096)
        return TK3D_ERR_UNSUPPORTED;
    return C < kRounded ? edge_forward(x, index, w, gamma, B, N, K, C, O, static_cast<double *>(workspace),
                                       extreme, (hipStream_t)stream)
                        : edge_forward(x, index, w, gamma, B, N, K, C, O, static_cast<float *>(workspace),
                                       extreme, (hipStream_t)stream);
}

int tk3d_mlp_edge_lists(const int64_t *index, int B, int N, int K, int32_t *lists, void *stream)
{
    if (!tk3d_mlp_edge_supported(B, N, K, 1))
        return TK3D_ERR_UNSUPPORTED;
    const int rc = tk_allow_dynamic_lds<edge_lists_kernel>(32768 * 4);
    if (rc != TK3D_OK)
        return rc;
    // eight slices of a batch element, as long as every workgroup has a CU and 64 points
    int slices = tk_cu_count() / B;
    slices = slices > 8 ? 8 : slices;
    slices = slices > N / 64 ? N / 64 : slices;
    slices = slices < 1 ? 1 : slices;
    const int own = (N + slices - 1) / slices;
    edge_lists_kernel<<<B * slices, 1024, own * 4, (hipStream_t)stream>>>(index, N, K, own, slices, lists);
    return tk_launch_status();
}

int64_t tk3d_mlp_edge_backward_bytes(int B, int N, int O, int C)
{
    const int64_t partial = (int64_t)weight_runs(B, N, O, C).parts * 2 * tiles_of(O) * kTile * C * 8;
    const int64_t points = (int64_t)B * N * 4;
    return partial + points * ((may_gather(N) ? 2 * O : 0) + 2 * O + 3 * (int64_t)C);
}

int tk3d_mlp_edge_backward_f32(const float *g, const float *extreme, const unsigned char *arg,
                               const float *x, const int64_t *index, const int32_t *lists, const float *w,
                               int B, int N, int K, int C, int O, const tk3d_mlp_norm *norm,
                               const float *coef, void *workspace, float *dx, float *dw, void *stream_)
{
    if (!tk3d_mlp_edge_supported(B, N, K, O) || C <= 0 || C > 4096)
        return TK3D_ERR_UNSUPPORTED;
    const hipStream_t stream = (hipStream_t)stream_;
    const WeightRuns r = weight_runs(B, N, O, C);
    const int half = tiles_of(O) * kTile;
    // the workspace: partial sums, sel [B, N, O] of 8 bytes if the sums may be gathered, duv [B, 2 O, N], rows [B, N,
    // C], st [B, 2 C, N]
    double *partial = reinterpret_cast<double *>(workspace);
    int2 *sel = reinterpret_cast<int2 *>(partial + (int64_t)r.parts * 2 * half * C);
    float *duv = reinterpret_cast<float *>(sel + (may_gather(N) ? (int64_t)B * N * O : 0));
    float *rows = duv + (int64_t)B * N * 2 * O, *st = rows + (int64_t)B * N * C;
    const int tiles = (N + kPoints - 1) / kPoints, blocks = (O + kChannels - 1) / kChannels;
    const int gathers = (N + kGather - 1) / kGather * B;
    int rc = TK3D_OK;
    // Few long rows are better off gathered (us of the whole backward, gathered and owned, 64 -> 64 channels, one
    // cloud of 16384 points 119.5, 128.1; of 8192 97.6, 98.1; of 6000 96.5, 93.0; of 2048 88.2, 77.2; 128 rows of
    // 16384 182.3, 174.8), as are rows that LDS does not hold. Two channels of a workgroup share the lines of the
    // neighbours, as long as that leaves every CU a workgroup (512 rows of 2048: 10.5 us, one channel 12.5).
    const int64_t channels = (int64_t)B * O;
    if (!may_gather(N) || (owners_lds(N, 1) <= kOwnersLds && channels * 2 >= tk_cu_count())) {
        const bool two = channels >= 2 * tk_cu_count() && owners_lds(N, 2) <= kOwnersLds;
        rc = two ? edge_owners<2>(g, extreme, arg, index, B, N, K, O, *norm, coef, duv, stream)
                 : edge_owners<1>(g, extreme, arg, index, B, N, K, O, *norm, coef, duv, stream);
        if (rc != TK3D_OK)
            return rc;
    } else {
        edge_select_kernel<<<dim3(tiles, blocks, B), kBlock, 0, stream>>>(g, extreme, arg, N, O, *norm, coef, sel);
        edge_sparse_kernel<<<dim3(gathers, blocks), kBlock, 0, stream>>>(sel, lists, B, N, K, O, duv);
    }
    edge_rows_kernel<<<dim3(tiles, (C + kChannels - 1) / kChannels, B), kBlock, 0, stream>>>(x, C, N, rows);
    if (C <= 4)
        edge_neighbours_kernel<4><<<dim3(gathers, 1), kBlock, 0, stream>>>(rows, index, lists, B, N, K, C, st);
    else if (C <= 16)
        edge_neighbours_kernel<16><<<dim3(gathers, 1), kBlock, 0, stream>>>(rows, index, lists, B, N, K, C,
                                                                             st);
    else
        edge_neighbours_kernel<64><<<dim3(gathers, (C + 63) / 64), kBlock, 0, stream>>>(rows, index, lists,
                                                                                        B, N, K, C, st);
    const EdgeGradOp grad{{}, x, st, w, coef, norm->mean, lists, duv, C, O, K, half, 2 * half, N};
    rc = launch_product(grad, B, stream);
    if (rc == TK3D_OK && dx) {
        const EdgeInputOp input{{}, duv, w, dx, O, C, N};
        rc = launch_product(input, B, stream);
    }
    if (rc != TK3D_OK)
        return rc;
    const EdgeWeightOp weight{{}, x, duv, partial, N, O, half, r.padded, r.run, r.total, 2 * half, C};
    rc = launch_product(weight, r.parts, stream);
    if (rc != TK3D_OK)
        return rc;
    edge_weight_sum_kernel<<<(2 * half * C + 15) / 16, kBlock, 0, stream>>>(partial, r.parts, half, O, C, dw);
    return tk_launch_status();
}

}  // extern "C"
