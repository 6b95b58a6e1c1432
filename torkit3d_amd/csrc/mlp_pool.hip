// Backward of a shared-MLP layer under a maximum: what is sparse in it (include/tk3d_mlp.h has the algebra,
// mlp_grad.hip and mlp_wide.hip the dense half), and the small products of its weights.
//
// In a group of S positions a channel o has one value a e, at one place, so that W^T (a e) and (a e) x^T take O x I
// operations a group. As products over all positions (matrix cores, zeros among the rows) they took S times as many.
#include "mlp_common.h"

namespace {

// ---- coefficients and the sparse gradient ----------------------------------------------------------------

struct PoolGradArgs {
    const float *g, *extreme;
    const unsigned char *arg;
    const int *arg32;
    int B, C, M, count;  // count = B * M
    tk3d_mlp_norm norm;
    double2 *partial;    // [C][slots], or NULL: a workgroup has the whole of its channel
};

// f(place in [B, C, M], y, g) for a workgroup's groups of its channel, four loads of either on their way together.
// (One by one, each behind the trip of the one before, the four launches of mlp_pool_grad_kernel in a PointNet++
// segmentation step took 47 us, 41 now, mlp_pool_sums_kernel 8.0, 5.9.)
template <typename F> __device__ __forceinline__ void for_groups(const PoolGradArgs &a, const F &f)
{
    constexpr int U = 4;
    const int step = gridDim.x * blockDim.x;
    for (int i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < a.count; i0 += U * step) {
        int64_t at[U];
        float y[U], g[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * step < a.count ? i0 + u * step : i0, b = i / a.M;
            at[u] = ((int64_t)b * a.C + blockIdx.y) * a.M + (i - b * a.M);
            y[u] = a.extreme[at[u]];
            g[u] = a.g[at[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * step < a.count)
                f(at[u], y[u], g[u]);
    }
}

__device__ __forceinline__ double2 pool_sums(const PoolGradArgs &a, f32x4 ss, double2 *lds)
{
    double2 v{0.0, 0.0};
    for_groups(a, [&](int64_t, float y, float g) {
        const float e = passes(normalised(y, ss)) ? g : 0.0f;
        v.x += e;
        v.y += (double)e * (double)(y - ss.x);
    });
    return block_sum(v, lds);
}

__global__ void __launch_bounds__(kBlock) mlp_pool_sums_kernel(PoolGradArgs a)
{
    __shared__ double2 lds[kWaves];
    const double2 v = pool_sums(a, constants_of(a.norm, blockIdx.y), lds);
    if (threadIdx.x == 0)
        a.partial[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = v;
}

__global__ void __launch_bounds__(1024)
    mlp_pool_grad_kernel(PoolGradArgs a, double n, const float *w, int I, tk3d_mlp_norm inner, bool shifted,
                         int2 *sel, float *coef, float *dgamma, float *dbeta)
{
    __shared__ double2 lds[16], lds2[16];
    const int c = blockIdx.y;
    const f32x4 ss = constants_of(a.norm, c);
    double2 wm{0.0, 0.0};
    for (int i = threadIdx.x; i < I; i += blockDim.x) {
        const f32x4 k = constants_of(inner, i);
        wm.x += (double)w[(int64_t)c * I + i] * (double)(shifted ? k.w : centre_of(k));
    }
    wm = block_sum(wm, lds2);
    const double2 sum = a.partial ? slot_sum(a.partial, gridDim.x, c, lds) : pool_sums(a, ss, lds);
    const Coefficients k = grad_coefficients(sum, n, a.norm, c, wm.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        reinterpret_cast<f32x4 *>(coef)[c] = k.abd;
        dgamma[c] = k.dgamma;
        dbeta[c] = k.dbeta;
    }
    for_groups(a, [&](int64_t j, float y, float g) {
        const float e = passes(normalised(y, ss)) ? g : 0.0f;
        sel[j] = int2{__float_as_int(k.abd.x * e), a.arg ? (int)a.arg[j] : a.arg32[j]};
    });
}

// ---- the sparse halves ------------------------------------------------------------------------------------

constexpr int kRow = 65;  // of a tile in LDS, for 64 channels

__device__ __forceinline__ float scalar_of(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

struct SparseArgs {
    const int2 *sel;       // [B, O, M]
    const float *w;        // [O][I] (scatter)
    const float *y;        // [B, I, P] (outer)
    tk3d_mlp_norm norm;    // of y
    float *out;            // [B, I, P] (scatter), partial sums [splits][O][I] (outer)
    int O, I, M, run;      // a wave takes `run` consecutive groups at once
    int units, total;      // runs: per batch element, in all
};

// out[b, i, (m, place)] = sum over o of w[o][i] a e; zero at the other places. A
// lane adds to a column of its own, in the order of o: 12 to 16 waves a CU cover the trips to LDS (as LDS
// atomics, without the trips, the additions took 341 us for 42 on 16 x 512 groups of 32). Neither four reads at
// once where four o have four places (50 us) nor the sums in registers indexed by the place (54 us) was faster.
template <int S>
__global__ void __launch_bounds__(kBlock) mlp_pool_scatter_kernel(SparseArgs a)
{
    extern __shared__ float tiles[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *tile = tiles + wave * (S * kRow);
    const int i0 = blockIdx.y * 64, c = i0 + lane < a.I ? i0 + lane : a.I - 1;
    const int p = lane & (S - 1), first = lane / S;  // of the loop over positions
    for (int unit = blockIdx.x * kWaves + wave; unit < a.total; unit += gridDim.x * kWaves) {
        const int b = unit / a.units, from = (unit - b * a.units) * a.run;
        const int to = from + a.run < a.M ? from + a.run : a.M;
        for (int m = from; m < to; ++m) {
#pragma unroll 8
            for (int q = 0; q < S; ++q)
                tile[q * kRow + lane] = 0.0f;
            for (int o0 = 0; o0 < a.O; o0 += 64) {
                const int o = o0 + lane < a.O ? o0 + lane : a.O - 1;
                const int2 s = a.sel[((int64_t)b * a.O + o) * a.M + m];
                const float e = o0 + lane < a.O ? __int_as_float(s.x) : 0.0f;
                const int n = a.O - o0 < 64 ? a.O - o0 : 64;
                for (int k = 0; k < n; k += 8) {
                    float w[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        w[j] = a.w[(int64_t)(o0 + (k + j < n ? k + j : n - 1)) * a.I + c];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {  // (lanes from n on: zeros at a place of the tile)
                        float &at = tiles[wave * (S * kRow) + __builtin_amdgcn_readlane(s.y, k + j) * kRow + lane];
                        at = __builtin_fmaf(scalar_of(e, k + j), w[j], at);
                    }
                }
            }
            tk_wave_fence();
            const int64_t P = (int64_t)a.M * S;
            float *out = a.out + ((int64_t)b * a.I + i0) * P + (int64_t)m * S + p;
#pragma unroll 8
            for (int i = first; i < 64; i += 64 / S)
                if (i0 + i < a.I)
                    out[i * P] = tile[p * kRow + i];
            tk_wave_fence();
        }
    }
}

// partial[split][o][i] = sum over groups of a e (relu(norm(y[i, (m, place)])) less the centre of i): 64 rows and 64
// columns a wave, rows in registers, the group's S x 64 activations in LDS (rows of 65: written by positions, read
// by channels). From 129 rows on four waves share a group, each normalises a quarter of it, and a workgroup of
// sixteen has all rows: with a group a wave the values were read and normalised once per 64 rows and two waves a
// SIMD waited for them (O = 256, I = 128, 2048 groups of 64 44 -> 30 us, O = 300, I = 33, 2050 groups of 32
// 35 -> 25 us; two waves on 65 to 128 rows 31 -> 33 us). The next group's values are requested before the present
// one's rows are added up; where they are shared they go to the other half of LDS.
template <int S, int WO>
__global__ void __launch_bounds__(WO * kBlock) mlp_pool_outer_kernel(SparseArgs a)
{
    constexpr int NW = WO * kWaves, GROUPS = NW / WO, HALVES = WO == 1 ? 1 : 2;
    constexpr int LOADS = S / WO, TILE = S * kRow;
    extern __shared__ float tiles[];
    __shared__ f32x4 constants[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot = wave / WO, share = wave % WO;
    float *tile = tiles + slot * (HALVES * TILE);
    const int o0 = (blockIdx.y * WO + share) * 64, i0 = blockIdx.z * 64;
    const int o = o0 + lane < a.O ? o0 + lane : a.O - 1;
    const int p = lane & (S - 1), first = lane / S + share * LOADS * (64 / S);
    if (tid < 64)
        constants[tid] = constants_of(a.norm, i0 + tid < a.I ? i0 + tid : a.I - 1);
    __syncthreads();
    float acc[64];
#pragma unroll
    for (int k = 0; k < 64; ++k)
        acc[k] = 0.0f;
    const int64_t P = (int64_t)a.M * S;
    float v[LOADS];
    int2 sel{0, 0};
    const auto load = [&](int b, int m) {
        sel = a.sel[((int64_t)b * a.O + o) * a.M + m];
        const float *y = a.y + (int64_t)b * a.I * P + (int64_t)m * S + p;
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            const int i = i0 + first + q * (64 / S);
            v[q] = y[(i < a.I ? i : a.I - 1) * P];
        }
    };
    const auto meet = [&] {  // the waves that share a group
        if constexpr (WO == 1) {
            tk_wave_fence();
        } else {
            __syncthreads();
        }
    };
    // Rounds of a group for every slot, as many as the first slot has, whose runs come first.
    const int step = gridDim.x * GROUPS;
    int unit = blockIdx.x * GROUPS + slot, b = unit / a.units, m = (unit - b * a.units) * a.run;
    bool mine = unit < a.total;
    int lead = blockIdx.x * GROUPS, rounds = 0;
    if constexpr (WO > 1)
        for (; lead < a.total; lead += step)
            rounds += a.run;
    if (mine)
        load(b, m);
    for (int round = 0; WO == 1 ? mine : round < rounds; ++round) {
        float *to = tile + (HALVES == 2 ? (round & 1) * TILE : 0);
        const bool add = WO == 1 || mine;
        if (add)
#pragma unroll
            for (int q = 0; q < LOADS; ++q) {
                const int i = first + q * (64 / S);
                to[p * kRow + i] = relu(normalised(v[q], constants[i])) - centre_of(constants[i]);
            }
        const float e = add && o0 + lane < a.O ? __int_as_float(sel.x) : 0.0f;
        const int place = sel.y & (S - 1);
        meet();
        if (add) {
            const int end = (unit - b * a.units + 1) * a.run;
            if (++m >= (end < a.M ? end : a.M)) {
                unit += step;
                b = unit / a.units;
                m = (unit - b * a.units) * a.run;
                mine = unit < a.total;
            }
            if (mine)
                load(b, m);
        }
        if (add)
#pragma unroll
            for (int k = 0; k < 64; ++k)
                acc[k] = __builtin_fmaf(scalar_of(e, k),
                                        to[__builtin_amdgcn_readlane(place, k) * kRow + lane], acc[k]);
        if constexpr (WO == 1)
            meet();
    }
    // (one slot after the other, WO times 16 KB)
    for (int w = 0; w < GROUPS; ++w) {
        __syncthreads();
        if (w == slot)
#pragma unroll
            for (int k = 0; k < 64; ++k) {
                float &sum = tiles[(share * 64 + k) * 64 + lane];
                sum = w ? sum + acc[k] : acc[k];
            }
    }
    __syncthreads();
    for (int e = tid; e < WO * 64 * 64; e += NW * 64) {
        const int row = blockIdx.y * (WO * 64) + (e >> 6), i = i0 + (e & 63);
        if (row < a.O && i < a.I)
            a.out[((int64_t)blockIdx.x * a.O + row) * a.I + i] = tiles[e];
    }
}

// ---- a group that is a whole row --------------------------------------------------------------------------------
//
// One value per channel and batch element: of a layer under a maximum over all points dy is dense only through b y
// + d, whose products are as wide as the layer's input and not as its output (1024 channels of 320, 8 x 2048
// points, both gradients and what led to them: 337 us dense, 216 us so; 1024 of 128, 32 x 2048 points, with its forward
// and backward in front 1216 -> 663).

// out[b, i, p] = sum over the o whose place is p of w[o][i] a e, in the order of o. A wave has 64 positions and 64
// channels: it looks through the places, and takes eight o of its own at once.
__global__ void __launch_bounds__(kBlock)
    mlp_rows_scatter_kernel(const int2 *sel, const float *w, int O, int I, int P, int tiles, int total, float *out)
{
    constexpr int AT_ONCE = 8;
    extern __shared__ float tiles_[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *tile = tiles_ + wave * (64 * kRow);
    const int i0 = blockIdx.y * 64, c = i0 + lane < I ? i0 + lane : I - 1;
    for (int unit = blockIdx.x * kWaves + wave; unit < total; unit += gridDim.x * kWaves) {
        const int b = unit / tiles, from = (unit - b * tiles) * 64;
#pragma unroll 8
        for (int q = 0; q < 64; ++q)
            tile[q * kRow + lane] = 0.0f;
        int2 next = sel[(int64_t)b * O + (lane < O ? lane : O - 1)];
        for (int o0 = 0; o0 < O; o0 += 64) {
            const int2 s = next;
            const int after = o0 + 64 + lane;
            next = sel[(int64_t)b * O + (after < O ? after : O - 1)];
            const float e = __int_as_float(s.x);
            unsigned long long mine =
                __ballot(o0 + lane < O && (unsigned)s.y < (unsigned)P && (unsigned)(s.y - from) < 64u);
            while (mine) {
                int at[AT_ONCE];
                float v[AT_ONCE];
                int n = 0;
#pragma unroll
                for (int j = 0; j < AT_ONCE; ++j) {
                    at[j] = mine ? __builtin_ctzll(mine) : at[0];
                    n += mine ? 1 : 0;
                    mine &= mine - 1;  // (zero stays zero)
                    v[j] = w[(int64_t)(o0 + at[j]) * I + c];
                }
#pragma unroll
                for (int j = 0; j < AT_ONCE; ++j)
                    if (j < n) {
                        float &sum = tile[(__builtin_amdgcn_readlane(s.y, at[j]) - from) * kRow + lane];
                        sum = __builtin_fmaf(scalar_of(e, at[j]), v[j], sum);
                    }
            }
        }
        tk_wave_fence();
        float *to = out + ((int64_t)b * I + i0) * P + from + lane;
#pragma unroll 8
        for (int i = 0; i < 64; ++i)
            if (i0 + i < I && from + lane < P)
                to[(int64_t)i * P] = tile[lane * kRow + i];
        tk_wave_fence();
    }
}

// dw[o][i] = sum over b of a e x', x' that of channel i at the place of o. Neighbouring lanes have neighbouring o,
// whose places are within one row of x: the row stays in L1 for all of them. One chain over the batch, in fp64: in
// fp32 4096 clouds of 16 points, 70 -> 160 channels, were twice as far from 64 bits as the stock modules.
template <bool SHIFTED>
__global__ void __launch_bounds__(kBlock) mlp_rows_outer_kernel(const int2 *sel, const float *x, tk3d_mlp_norm norm, int B,
                                                                int O, int I, int P, float *dw)
{
    const int i = blockIdx.x, o = blockIdx.y * kBlock + threadIdx.x;
    const f32x4 k = constants_of(norm, i);
    if (o >= O)
        return;
    double sum = 0.0;
#pragma unroll 4
    for (int b = 0; b < B; ++b) {
        const int2 s = sel[(int64_t)b * O + o];
        const float v = x[((int64_t)b * I + i) * P + ((unsigned)s.y < (unsigned)P ? s.y : 0)];
        sum = __builtin_fma((double)__int_as_float(s.x),
                            (double)(SHIFTED ? v - k.w : relu(normalised(v, k)) - centre_of(k)), sum);
    }
    dw[(int64_t)o * I + i] = (float)sum;
}

// mean[c], a workgroup a channel. (Where a sum is counted from need not be known to the last bit.)
__global__ void __launch_bounds__(kBlock) mlp_channel_means_kernel(const float *x, int B, int C, int P, float *mean)
{
    __shared__ double2 lds[kWaves];
    const int c = blockIdx.x;
    float sum = 0.0f;
    for (int b = 0; b < B; ++b)
#pragma unroll 8
        for (int i = threadIdx.x; i < P; i += kBlock)
            sum += x[((int64_t)b * C + c) * P + i];
    const double2 s = block_sum(double2{sum, 0.0}, lds);
    if (threadIdx.x == 0)
        mean[c] = (float)(s.x / ((double)B * P));
}

// ---- small products of the weights -----------------------------------------------------------------------
//
// A tile of results a workgroup on the matrix cores, the sum shared by its four waves: these are chains of trips to
// L2 (in tiles of 16 x 16 through LDS, two barriers per 16 of the sum, gram took 19 us on O = 512, I = 256; in fp32 on the
// matrix cores 14.5, in fp64 8.5).

constexpr int kStep = 16, kStepGrad = 8;  // steps of four of the sum that are requested at once

typedef double f64x4 __attribute__((ext_vector_type(4)));

// The four waves' sums of a tile of 16 x 16 added up: wave r returns the result in row 4 r + lane / 16.
__device__ __forceinline__ double add_up(const f64x4 &sum, double (*lds)[4][64], int wave, int lane)
{
#pragma unroll
    for (int r = 0; r < 4; ++r)
        lds[wave][r][lane] = sum[r];
    __syncthreads();
    return (lds[0][wave][lane] + lds[1][wave][lane]) + (lds[2][wave][lane] + lds[3][wave][lane]);
}

// gram[k][c] = sum_o W[o][k] b[o] W[o][c]; the first row of blocks also adds up bias[c]. In fp64, rounded once: an
// error here is the same at all positions, and what is added up over them next, the gradients of the batch norm in
// front, is small (dbeta under a maximum over 2048 points from sums in fp32 twice as far from 64 bits as from a
// dense backward, now no farther).
__global__ void __launch_bounds__(kBlock)
    mlp_pool_gram_kernel(const float *w, const float *coef, int O, int I, float *gram, float *bias)
{
    __shared__ double lds[kWaves][4][64], part[kWaves][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, quarter = lane >> 4, l16 = lane & 15;
    const int k = blockIdx.y * 16 + l16, c = blockIdx.x * 16 + l16;
    const int kk = k < I ? k : I - 1, cc = c < I ? c : I - 1;
    f64x4 sum{0.0, 0.0, 0.0, 0.0};
    double off = 0.0;
    for (int o0 = wave * (4 * kStep); o0 < O; o0 += kWaves * 4 * kStep) {
        float x[kStep], y[kStep], b[kStep], d[kStep];
#pragma unroll
        for (int s = 0; s < kStep; ++s) {
            const int o = o0 + 4 * s + quarter, at = o < O ? o : O - 1;
            x[s] = w[(int64_t)at * I + kk];
            y[s] = w[(int64_t)at * I + cc];
            b[s] = o < O ? coef[at * 4 + 1] : 0.0f;
            d[s] = o < O ? coef[at * 4 + 2] : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < kStep; ++s) {
            sum = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x[s] * (double)b[s], (double)y[s], sum, 0, 0, 0);
            off = __builtin_fma((double)d[s], (double)y[s], off);
        }
    }
    off += __shfl_xor(off, 16);
    off += __shfl_xor(off, 32);
    if (quarter == 0)
        part[wave][l16] = off;
    const double total = add_up(sum, lds, wave, lane);
    const int row = blockIdx.y * 16 + 4 * wave + quarter;
    if (row < I && c < I)
        gram[(int64_t)row * I + c] = (float)total;
    if (blockIdx.y == 0 && threadIdx.x < 16 && c < I)
        bias[c] = (float)((part[0][l16] + part[1][l16]) + (part[2][l16] + part[3][l16]));
}

// dw[o][i] += b[o] (W xx)[o][i] + d[o] xsum[i], terms of which the sum is a small part: in fp64 as well
__global__ void __launch_bounds__(kBlock)
    mlp_pool_weight_grad_kernel(const float *w, const float *coef, const float *xx, const float *xsum,
                                int O, int I, float *dw)
{
    __shared__ double lds[kWaves][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, quarter = lane >> 4, l16 = lane & 15;
    const int o = blockIdx.y * 16 + l16, i = blockIdx.x * 16 + l16, ii = i < I ? i : I - 1;
    const float *row = w + (int64_t)(o < O ? o : O - 1) * I;
    f64x4 sum{0.0, 0.0, 0.0, 0.0};
    for (int k0 = wave * (4 * kStepGrad); k0 < I; k0 += kWaves * 4 * kStepGrad) {
        float x[kStepGrad], y[kStepGrad];
#pragma unroll
        for (int s = 0; s < kStepGrad; ++s) {
            const int k = k0 + 4 * s + quarter, at = k < I ? k : I - 1;
            x[s] = k < I ? row[at] : 0.0f;
            y[s] = k < I ? xx[(int64_t)(at < ii ? at : ii) * I + (at < ii ? ii : at)] : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < kStepGrad; ++s)
            sum = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x[s], (double)y[s], sum, 0, 0, 0);
    }
    const double total = add_up(sum, lds, wave, lane);
    const int to = blockIdx.y * 16 + 4 * wave + quarter;
    if (to < O && i < I) {
        float &out = dw[(int64_t)to * I + i];
        out = (float)__builtin_fma((double)coef[to * 4 + 1], total,
                                   __builtin_fma((double)coef[to * 4 + 2], (double)xsum[i], (double)out));
    }
}

// ---- launches ----------------------------------------------------------------------------------------------

// Runs of four groups read whole sectors of sel ([B, O, M]), as long as every SIMD keeps a wave.
int outer_run(int B, int M) { return (int64_t)B * M >= 16 * tk_cu_count() ? 4 : 1; }

void fill_sparse(SparseArgs &a, int B, int run)
{
    a.run = run;
    a.units = (a.M + a.run - 1) / a.run;
    a.total = B * a.units;
}


// Workgroups to a channel, 1024 groups each, from 8192 groups on; below, one, and one launch. (64 channels of
// 16384 groups 18 -> 11.5 us, 128 of 8192 12.4 -> 11.5; 256 of 2048 7.6 for 9.7.)
int grad_slots(int B, int C, int M)
{
    const int64_t groups = (int64_t)B * M, most = (8 * tk_cu_count() + C - 1) / C;
    const int64_t slots = groups < 8192 ? 1 : (groups + 1023) / 1024;
    return (int)(slots < most ? slots : most);
}

// Waves that share a group in mlp_pool_outer_kernel.
int sharing(int O) { return O > 128 ? 4 : 1; }

template <int S, int WO> int launch_outer(const SparseArgs &a, int splits, hipStream_t stream)
{
    constexpr int tiles = kWaves * (WO == 1 ? 1 : 2) * S * kRow * 4, sums = WO * 64 * 64 * 4;
    constexpr int bytes = tiles > sums ? tiles : sums;
    static_assert(bytes <= 160 << 10, "LDS of a CU");
    const int rc = tk_allow_dynamic_lds<mlp_pool_outer_kernel<S, WO>>(bytes);
    if (rc != TK3D_OK)
        return rc;
    const dim3 grid(splits, (a.O + 64 * WO - 1) / (64 * WO), (a.I + 63) / 64);
    mlp_pool_outer_kernel<S, WO><<<grid, WO * kBlock, bytes, stream>>>(a);
    return tk_launch_status();
}

template <int S> int launch_outer(const SparseArgs &a, int splits, hipStream_t stream)
{
    return sharing(a.O) == 1 ? launch_outer<S, 1>(a, splits, stream) : launch_outer<S, 4>(a, splits, stream);
}

}  // namespace

extern "C" {

int tk3d_mlp_pool_grad_slots(int B, int C, int M) { return grad_slots(B, C, M); }

int tk3d_mlp_pool_grad_f32(const float *g, const float *extreme, const unsigned char *arg,
                           const int32_t *arg32, int B, int C, int M, int64_t positions, const tk3d_mlp_norm *norm, const float *w,
                           int I, const tk3d_mlp_norm *inner, int shifted, void *partial, void *sel,
                           float *coef, float *dgamma, float *dbeta, void *stream_)
{
    if (B <= 0 || C <= 0 || M <= 0 || I <= 0)
        return TK3D_ERR_BAD_SIZE;
    if (!tk_fits(TK_MAX_I32 - (1 << 24), B, M) || C > 65535)
        return TK3D_ERR_UNSUPPORTED;
    const dim3 grid(grad_slots(B, C, M), C);
    const PoolGradArgs a{g, extreme, arg, arg32, B, C, M, B * M, *norm,
                         grid.x > 1 ? reinterpret_cast<double2 *>(partial) : nullptr};
    const hipStream_t stream = (hipStream_t)stream_;
    if (grid.x > 1) {
        mlp_pool_sums_kernel<<<grid, kBlock, 0, stream>>>(a);
        const int rc = tk_launch_status();
        if (rc != TK3D_OK)
            return rc;
    }
    mlp_pool_grad_kernel<<<grid, grid.x > 1 || a.count <= 1024 ? kBlock : 1024, 0, stream>>>(
        a, (double)positions, w, I, *inner, shifted != 0, reinterpret_cast<int2 *>(sel), coef, dgamma, dbeta);
    return tk_launch_status();
}

int tk3d_mlp_pool_scatter_f32(const void *sel, const float *w, int B, int O, int I, int M, int group,
                              float *out, void *stream_)
{
    if (B <= 0 || O <= 0 || I <= 0 || M <= 0)
        return TK3D_ERR_BAD_SIZE;
    if ((group != 32 && group != 64) || !tk_fits(TK_MAX_I32, B, M) || I > 65535 * 64)
        return TK3D_ERR_UNSUPPORTED;
    SparseArgs a{};
    a.sel = reinterpret_cast<const int2 *>(sel);
    a.w = w;
    a.out = out;
    a.O = O;
    a.I = I;
    a.M = M;
    // Groups in a row share the lines of `sel` they come from, but a launch that leaves lanes idle for it
    // loses more: as many as the resident waves (16 of a CU, 8 with 64 places, by LDS) have rounds for, up to
    // four. us, four of them from 4096 groups on, and now: O = 128, I = 64, 8 x 512 groups of 32 38, 19; 16 x
    // 512 46, 34 (two); 32 x 512 63, 63 (four; one 66); O = 256, I = 128, 16 x 128 groups of 64 48, 46.
    const int64_t waves = (int64_t)B * M * ((I + 63) / 64);
    const int64_t rounds = waves / ((group == 32 ? 16 : 8) * (int64_t)tk_cu_count());
    fill_sparse(a, B, rounds >= 4 ? 4 : rounds >= 2 ? 2 : 1);
    const int bytes = kWaves * group * kRow * 4;
    const int rc = group == 32 ? tk_allow_dynamic_lds<mlp_pool_scatter_kernel<32>>(bytes)
                               : tk_allow_dynamic_lds<mlp_pool_scatter_kernel<64>>(bytes);
    if (rc != TK3D_OK)
        return rc;
    const int wgs = (a.total + kWaves - 1) / kWaves, most = 4 * tk_cu_count();
    const dim3 grid(wgs < most ? wgs : most, (I + 63) / 64);
    if (group == 32)
        mlp_pool_scatter_kernel<32><<<grid, kBlock, bytes, (hipStream_t)stream_>>>(a);
    else
        mlp_pool_scatter_kernel<64><<<grid, kBlock, bytes, (hipStream_t)stream_>>>(a);
    return tk_launch_status();
}

// Two workgroups of four waves to a CU, or one of sixteen, and no more than there are runs for.
int tk3d_mlp_pool_outer_splits(int B, int O, int I, int M)
{
    SparseArgs a{};
    a.M = M;
    fill_sparse(a, B, outer_run(B, M));
    const int wo = sharing(O);
    const int blocks = ((O + 64 * wo - 1) / (64 * wo)) * ((I + 63) / 64), wgs = (a.total + kWaves - 1) / kWaves;
    const int most = ((wo == 1 ? 2 : 1) * tk_cu_count() + blocks - 1) / blocks;
    return wgs < most ? wgs : most;
}

int tk3d_mlp_pool_outer_f32(const void *sel, const float *y, const tk3d_mlp_norm *norm, int B, int O,
                            int I, int M, int group, float *partial, void *stream_)
{
    if (B <= 0 || O <= 0 || I <= 0 || M <= 0)
        return TK3D_ERR_BAD_SIZE;
    if ((group != 32 && group != 64) || !tk_fits(TK_MAX_I32, B, M) || I > 65535 * 64 || O > 65535 * 64)
        return TK3D_ERR_UNSUPPORTED;
    SparseArgs a{};
    a.sel = reinterpret_cast<const int2 *>(sel);
    a.y = y;
    a.norm = *norm;
    a.out = partial;
    a.O = O;
    a.I = I;
    a.M = M;
    fill_sparse(a, B, outer_run(B, M));
    const int splits = tk3d_mlp_pool_outer_splits(B, O, I, M);
    return group == 32 ? launch_outer<32>(a, splits, (hipStream_t)stream_)
                       : launch_outer<64>(a, splits, (hipStream_t)stream_);
}

int tk3d_mlp_rows_scatter_f32(const void *sel, const float *w, int B, int O, int I, int P, float *out, void *stream)
{
    if (B <= 0 || O <= 0 || I <= 0 || P <= 0)
        return TK3D_ERR_BAD_SIZE;
    const int tiles = (P + 63) / 64;
    if (!tk_fits(1 << 30, B, tiles) || I > 65535 * 64)
        return TK3D_ERR_UNSUPPORTED;
    constexpr int bytes = kWaves * 64 * kRow * 4;
    const int rc = tk_allow_dynamic_lds<mlp_rows_scatter_kernel>(bytes);
    if (rc != TK3D_OK)
        return rc;
    const int wgs = (B * tiles + kWaves - 1) / kWaves, most = 4 * tk_cu_count();
    mlp_rows_scatter_kernel<<<dim3(wgs < most ? wgs : most, (I + 63) / 64), kBlock, bytes, (hipStream_t)stream>>>(
        reinterpret_cast<const int2 *>(sel), w, O, I, P, tiles, B * tiles, out);
    return tk_launch_status();
}

int tk3d_mlp_rows_outer_f32(const void *sel, const float *x, int shifted, const tk3d_mlp_norm *norm, int B, int O,
                            int I, int P, float *dw, void *stream_)
{
    if (B <= 0 || O <= 0 || I <= 0 || P <= 0)
        return TK3D_ERR_BAD_SIZE;
    const dim3 grid(I, (O + kBlock - 1) / kBlock);
    const hipStream_t stream = (hipStream_t)stream_;
    if (shifted)
        mlp_rows_outer_kernel<true><<<grid, kBlock, 0, stream>>>(reinterpret_cast<const int2 *>(sel), x, *norm, B, O, I, P, dw);
    else
        mlp_rows_outer_kernel<false><<<grid, kBlock, 0, stream>>>(reinterpret_cast<const int2 *>(sel), x, *norm, B, O, I, P, dw);
    return tk_launch_status();
}

int tk3d_mlp_channel_means_f32(const float *x, int B, int C, int P, float *mean, void *stream)
{
    mlp_channel_means_kernel<<<C, kBlock, 0, (hipStream_t)stream>>>(x, B, C, P, mean);
    return tk_launch_status();
}

int tk3d_mlp_pool_gram_f32(const float *w, const float *coef, int O, int I, float *gram, float *bias,
                           void *stream)
{
    const int n = (I + 15) / 16;
    mlp_pool_gram_kernel<<<dim3(n, n), kBlock, 0, (hipStream_t)stream>>>(w, coef, O, I, gram, bias);
    return tk_launch_status();
}

int tk3d_mlp_pool_weight_grad_f32(const float *sparse, int sparse_splits, const float *xx,
                                  const float *xsum, int xx_splits, const float *w,
                                  const float *coef, int O, int I, float *scratch, float *dw,
                                  void *stream)
{
    const tk3d_mlp_sum sums[3] = {
        {sparse, dw, (int64_t)O * I, sparse_splits, O, I, I},
        {xx, scratch, (int64_t)I * I, xx_splits, I, I, I},
        {xsum, scratch + (int64_t)I * I, I, xx_splits, 1, I, I}};
    const int rc = tk3d_mlp_sum_f32(sums, 3, stream);
    if (rc != TK3D_OK)
        return rc;
    mlp_pool_weight_grad_kernel<<<dim3((I + 15) / 16, (O + 15) / 16), kBlock, 0, (hipStream_t)stream>>>(
        w, coef, scratch, scratch + (int64_t)I * I, O, I, dw);
    return tk_launch_status();
}

}  // extern "C"
