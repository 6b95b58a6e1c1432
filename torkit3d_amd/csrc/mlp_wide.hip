// Backward products of layers too wide for mlp_grad.hip, from tiles in LDS (entry points in mlp.hip).
//
// What bounds them: the fp32 matrix rate, if the operands get there. The kernels of mlp.hip bring rows straight
// from memory into the lanes: at 1024 channels every lane reads runs of a row of its own (64 cache lines a
// load) and every wave the whole of its operands through L1. Here a workgroup of eight waves shares a tile of
// either operand, read in whole lines and normalised once, in LDS: the next tile is on its way in registers while
// one is multiplied. Workgroups that read the same positions sit on one XCD, side by side in time. Chains are
// those of a tile or chunk, added up on top of each other.
//
// us, before -> now (TFLOP/s of the matrix rate's 157): weight gradient of 320 -> 1024 channels, 16384 positions
// 217 -> 120 (90), of 512 -> 1024, 2048 positions 38 -> 28 (77), of 256 -> 256, 1024 positions 14.5 -> 5.8; input
// gradient of 320 -> 1024, 16384 positions 165 -> 124 (87), of 320 -> 256 45 -> 36 (75). Activations times
// themselves (the dense half under a maximum), 320 x 320 on 16384 positions: 63 us, 42 without the blocks below
// the diagonal. Errors against 64 bits: dW 4.4e-7 -> 1.6e-7, dx 2.9e-7 -> 1.3e-7 of the result for the first.
#include "mlp_common.h"
#include "mlp_wide.h"

namespace {

constexpr int kWide = 512, kWideWaves = kWide / TK_WAVE;
constexpr int kWidePositions = 128;  // of the product's workgroups

__device__ __forceinline__ f32x4 read(const float *base, unsigned offset)
{
    return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(base) + offset);
}

// Linear workgroup `at` of groups x members: the members of a group follow each other on one XCD (workgroups
// go to the eight XCDs in turn).
__device__ __forceinline__ bool place_of(int at, int groups, int members, int &group, int &member)
{
    const int turn = at / 8;
    group = turn / members * 8 + at % 8;
    member = turn % members;
    return group < groups;
}
int placed(int groups, int members) { return (groups + 7) / 8 * 8 * members; }

// ---- the weight gradient: 128 rows and 64 columns a workgroup, two workgroups a CU --------------------------

struct WideOuterArgs {
    tk3d_mlp_outer p;
    int tiles, total;  // tiles of 32 positions: per batch element, in all
    int splits, rblocks, cblocks;
};

template <int ROW, int COL>
__global__ void __launch_bounds__(kWide, 4) mlp_wide_outer_kernel(WideOuterArgs a)
{
    constexpr int NP = 32, STRIDE = NP + 4, RB = 4, CB = 2;
    constexpr int STEP = kWide / 8, RL = 32 * RB / STEP, CL = 32 * CB / STEP;  // 16-byte loads of a thread, rows apart
    constexpr int ROWS = 32 * RB * STRIDE, HALF = ROWS + 32 * CB * STRIDE;
    constexpr bool kGrad = ROW == TK3D_MLP_ROW_GRAD || ROW == TK3D_MLP_ROW_GRAD_OUT;
    constexpr bool kRowSums = ROW == TK3D_MLP_ROW_CENTRED || ROW == TK3D_MLP_ROW_SHIFTED;
    __shared__ __attribute__((aligned(16))) float lds[2 * HALF];
    const tk3d_mlp_outer &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    const int R = p.row.K, C = p.col.K, P = p.P;
    int group, cblock;
    if (!place_of(blockIdx.x, a.splits * a.rblocks, a.cblocks, group, cblock))
        return;
    if (kRowSums && 2 * (group % a.rblocks) > cblock)  // (symmetric: nothing below the diagonal is read)
        return;
    const int split = group / a.rblocks, rbase = group % a.rblocks * (32 * RB), cbase = cblock * (32 * CB);

    // A thread's 16 bytes of every 64th row, and these rows' constants.
    const int quad = tid % 8, first = tid / 8;
    f32x4 x[RL], y[kGrad ? RL : 1], c[CL], coef[RL], row_act[RL], col_act[CL];
#pragma unroll
    for (int i = 0; i < RL; ++i) {
        const int r = rbase + first + i * STEP, row = r < R ? r : R - 1;
        if constexpr (kGrad)
            coef[i] = reinterpret_cast<const f32x4 *>(p.row.coef)[row];
        if constexpr (ROW == TK3D_MLP_ROW_GRAD_OUT || ROW == TK3D_MLP_ROW_CENTRED || ROW == TK3D_MLP_ROW_SHIFTED)
            row_act[i] = constants_of(p.row_norm, row);
    }
#pragma unroll
    for (int i = 0; i < CL; ++i) {
        const int r = cbase + first + i * STEP;
        if constexpr (COL != TK3D_MLP_COL_RAW)
            col_act[i] = constants_of(p.col_norm, r < C ? r : C - 1);
    }
    const auto load = [&](int tile) {
        const int b = tile / a.tiles, pos = (tile - b * a.tiles) * NP + 4 * quad;
        const unsigned at = pos < P ? pos : P - 4;
        const float *rx = p.row.x + (int64_t)b * p.row.batch_stride, *ry = p.row.y + (int64_t)b * p.row.batch_stride;
        const float *cx = p.col.x + (int64_t)b * p.col.batch_stride;
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const int r = rbase + first + i * STEP;
            const unsigned offset = ((unsigned)(r < R ? r : R - 1) * (unsigned)P + at) * 4u;
            x[i] = read(rx, offset);
            if constexpr (kGrad)
                y[i] = read(ry, offset);
        }
#pragma unroll
        for (int i = 0; i < CL; ++i) {
            const int r = cbase + first + i * STEP;
            c[i] = read(cx, ((unsigned)(r < C ? r : C - 1) * (unsigned)P + at) * 4u);
        }
    };
    // Positions past the last one are zero on either side.
    const auto store = [&](int tile, float *to) {
        const int b = tile / a.tiles;
        const bool in = (tile - b * a.tiles) * NP + 4 * quad < P;
        to += first * STRIDE + 4 * quad;
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float g = x[i][j];
                if constexpr (ROW == TK3D_MLP_ROW_GRAD_OUT)
                    g = passes(normalised(y[kGrad ? i : 0][j], row_act[i])) ? g : 0.0f;
                if constexpr (kGrad)
                    g = __builtin_fmaf(coef[i].x, g, __builtin_fmaf(coef[i].y, y[kGrad ? i : 0][j], coef[i].z));
                if constexpr (ROW == TK3D_MLP_ROW_CENTRED)
                    g = relu(normalised(g, row_act[i])) - centre_of(row_act[i]);
                if constexpr (ROW == TK3D_MLP_ROW_SHIFTED)
                    g -= centre_of(row_act[i]);
                v[j] = in ? g : 0.0f;
            }
            *reinterpret_cast<f32x4 *>(to + i * STEP * STRIDE) = v;
        }
#pragma unroll
        for (int i = 0; i < CL; ++i) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float h = c[i][j];
                if constexpr (COL == TK3D_MLP_COL_ACT || COL == TK3D_MLP_COL_CENTRED)
                    h = relu(normalised(h, col_act[i]));
                if constexpr (COL == TK3D_MLP_COL_CENTRED || COL == TK3D_MLP_COL_SHIFTED)
                    h -= centre_of(col_act[i]);
                v[j] = in ? h : 0.0f;
            }
            *reinterpret_cast<f32x4 *>(to + ROWS + i * STEP * STRIDE) = v;
        }
    };

    // A wave's 32 x 32 sums of a tile go on top of those of the tiles before it.
    const int wrow = wave / CB * 32, wcol = wave % CB * 32;
    tk_f32x16 total;
    float row_total = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        total[r] = 0.0f;
    const auto multiply = [&](const float *from) {
        tk_f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            acc[r] = 0.0f;
        const float *rows = from + (wrow + l32) * STRIDE + 4 * half;
        const float *columns = from + ROWS + (wcol + l32) * STRIDE + 4 * half;
        float row_sum = 0.0f;
        f32x4 g[2], h[2];
        const auto fetch = [&](int step) {
            g[step & 1] = *reinterpret_cast<const f32x4 *>(rows + 8 * step);
            h[step & 1] = *reinterpret_cast<const f32x4 *>(columns + 8 * step);
        };
        fetch(0);
#pragma unroll
        for (int step = 0; step < NP / 8; ++step) {
            if (step + 1 < NP / 8)
                fetch(step + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (kRowSums)
                    row_sum += g[step & 1][k];
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(g[step & 1][k], h[step & 1][k], acc, 0, 0, 0);
            }
        }
        row_total += row_sum;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            total[r] += acc[r];
    };

    load(split);  // (no more splits than there are tiles)
    store(split, lds);
    __syncthreads();
    for (int tile = split, now = 0; tile < a.total; tile += a.splits, now ^= 1) {
        const bool more = tile + a.splits < a.total;
        if (more)
            load(tile + a.splits);
        multiply(lds + now * HALF);
        if (more)
            store(tile + a.splits, lds + (now ^ 1) * HALF);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = rbase + wrow + 8 * (r >> 2) + 4 * half + (r & 3), column = cbase + wcol + l32;
        if (row < R && column < C)
            p.partial[((int64_t)split * R + row) * C + column] = total[r];
    }
    if constexpr (kRowSums) {
        row_total += __shfl_xor(row_total, 32);
        const int row = rbase + wrow + l32;
        if (p.rowsum && cbase == rbase && wave % CB == 0 && half == 0 && row < R)
            p.rowsum[(int64_t)split * R + row] = row_total;
    }
}

// ---- the product: 128 positions and 32 * CT channels a workgroup, one workgroup a CU -----------------------
//
// A wave has 32 positions and all CT tiles of channels; two teams of four waves share the input channels of
// every chunk of 32, and their sums meet in LDS at the end. CT is chosen so that it divides the layer's channels.

struct WideProductArgs {
    tk3d_mlp_product p;
    int tiles, groups;  // blocks of positions: per batch element, in all
    int cblocks, chunks;
    int rows4;          // weight rows are 16-byte aligned runs along the output channels
};

template <int IN, int OUT, int CT>
__global__ void __launch_bounds__(kWide) mlp_wide_product_kernel(WideProductArgs a)
{
    constexpr int KS = 2, PW = kWideWaves / KS, NP = kWidePositions, KC = 32;
    constexpr int GS = NP + 4, WS = 32 * CT + 4;              // strides of a channel's row in LDS
    constexpr int G = KC * GS, HALF = G + KC * WS;
    constexpr int QUADS = NP / 4, STEP = kWide / QUADS, GL = KC / STEP;
    constexpr int WQUADS = 8 * CT, WL = (KC * WQUADS + kWide - 1) / kWide;
    constexpr bool kGrad = IN == TK3D_MLP_IN_GRAD || IN == TK3D_MLP_IN_GRAD_OUT;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const tk3d_mlp_product &p = a.p;
    const tk3d_mlp_source &s = p.src[0];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    const int P = p.P, K = s.K, C = p.C;
    int group, cblock;
    if (!place_of(blockIdx.x, a.groups, a.cblocks, group, cblock))
        return;
    const int b = group / a.tiles, base = (group - b * a.tiles) * NP, cbase = cblock * (32 * CT);

    // The input channels' constants.
    f32x4 *grad_coef = reinterpret_cast<f32x4 *>(lds + 2 * HALF);
    f32x4 *act_coef = grad_coef + (kGrad ? a.chunks * KC : 0);
    for (int k = tid; k < a.chunks * KC; k += kWide) {
        const int row = k < K ? k : K - 1;
        if constexpr (kGrad)
            grad_coef[k] = reinterpret_cast<const f32x4 *>(s.coef)[row];
        if constexpr (IN != TK3D_MLP_IN_GRAD)
            act_coef[k] = constants_of(p.in_norm, row);
    }
    __syncthreads();

    const int quad = tid % QUADS, first = tid / QUADS;
    const bool in = base + 4 * quad < P;
    const unsigned at = in ? base + 4 * quad : P - 4;
    const float *sx = s.x + (int64_t)b * s.batch_stride, *sy = s.y + (int64_t)b * s.batch_stride;
    f32x4 x[GL], y[kGrad ? GL : 1], w[WL];
    const auto load = [&](int chunk) {
#pragma unroll
        for (int i = 0; i < GL; ++i) {
            const int k = chunk * KC + first + i * STEP;
            const unsigned offset = ((unsigned)(k < K ? k : K - 1) * (unsigned)P + at) * 4u;
            x[i] = read(sx, offset);
            if constexpr (kGrad)
                y[i] = read(sy, offset);
        }
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int e = tid + i * kWide, k = chunk * KC + e / WQUADS, c = cbase + 4 * (e % WQUADS);
            const float *row = s.w + (int64_t)(k < K ? k : K - 1) * s.wk;
            if (a.rows4) {  // (C is a multiple of four)
                w[i] = *reinterpret_cast<const f32x4 *>(row + (c < C ? c : C - 4));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    w[i][j] = row[(int64_t)(c + j < C ? c + j : C - 1) * s.wc];
            }
        }
    };
    // Input channels and positions past the last ones are zero; results of the surplus channels are dropped.
    const auto store = [&](int chunk, float *to) {
#pragma unroll
        for (int i = 0; i < GL; ++i) {
            const int k = chunk * KC + first + i * STEP;
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float g = x[i][j];
                if constexpr (IN == TK3D_MLP_IN_GRAD_OUT)
                    g = passes(normalised(y[kGrad ? i : 0][j], act_coef[k])) ? g : 0.0f;
                if constexpr (kGrad)
                    g = __builtin_fmaf(grad_coef[k].x, g,
                                       __builtin_fmaf(grad_coef[k].y, y[kGrad ? i : 0][j], grad_coef[k].z));
                else if constexpr (IN == TK3D_MLP_IN_CENTRED)
                    g = relu(normalised(g, act_coef[k])) - centre_of(act_coef[k]);
                else
                    g -= centre_of(act_coef[k]);
                v[j] = in && k < K ? g : 0.0f;
            }
            *reinterpret_cast<f32x4 *>(to + (first + i * STEP) * GS + 4 * quad) = v;
        }
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int e = tid + i * kWide, k = e / WQUADS;
            if (KC * WQUADS % kWide == 0 || k < KC)
                *reinterpret_cast<f32x4 *>(to + G + k * WS + 4 * (e % WQUADS)) =
                    chunk * KC + k < K ? w[i] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };

    // Sums of a chunk on top of those of the chunks before it.
    const int team = wave / PW, positions = wave % PW * 32;
    tk_f32x16 total[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            total[j][r] = 0.0f;
    const auto multiply = [&](const float *from) {
        constexpr int STEPS = KC / KS / 2;
        tk_f32x16 acc[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[j][r] = 0.0f;
        const int k0 = team * (KC / KS) + half;
        const float *gs = from + k0 * GS + positions + l32, *ws = from + G + k0 * WS + l32;
        float g[2], v[2][CT];
        const auto fetch = [&](int step) {
            g[step & 1] = gs[2 * step * GS];
#pragma unroll
            for (int j = 0; j < CT; ++j)
                v[step & 1][j] = ws[2 * step * WS + j * 32];
        };
        fetch(0);
#pragma unroll
        for (int step = 0; step < STEPS; ++step) {
            if (step + 1 < STEPS)
                fetch(step + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < CT; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(g[step & 1], v[step & 1][j], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                total[j][r] += acc[j][r];
    };

    load(0);
    store(0, lds);
    __syncthreads();
    for (int chunk = 0; chunk < a.chunks; ++chunk) {
        if (chunk + 1 < a.chunks)
            load(chunk + 1);
        multiply(lds + (chunk & 1) * HALF);
        if (chunk + 1 < a.chunks)
            store(chunk + 1, lds + (~chunk & 1) * HALF);
        __syncthreads();
    }

    // A tile of channels after the other: team t finishes its share of the runs of four positions.
    f32x4 *sums = reinterpret_cast<f32x4 *>(lds);  // [wave][4][64]
    constexpr int RUNS = 4 / KS;
    double sum1[CT], sum2[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        if (j)
            __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            sums[(wave * 4 + q) * 64 + lane] =
                f32x4{total[j][4 * q], total[j][4 * q + 1], total[j][4 * q + 2], total[j][4 * q + 3]};
        __syncthreads();
        const int channel = cbase + j * 32 + l32, c = channel < C ? channel : C - 1;
        const float bias = p.bias ? p.bias[c] : 0.0f;
        f32x4 norm{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (OUT == TK3D_MLP_OUT_MASK)
            norm = constants_of(p.out_norm, c);
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
            const int q = team * RUNS + i, pos = base + positions + 8 * q + 4 * half;
            f32x4 v = sums[(wave % PW * 4 + q) * 64 + lane] + sums[((PW + wave % PW) * 4 + q) * 64 + lane];
            const bool inside = pos < P;
            const int64_t offset = ((int64_t)b * C + c) * P + (inside ? pos : P - 4);
            v += bias;
            if constexpr (!kGrad)
                v += *reinterpret_cast<const f32x4 *>(p.add + offset);
            if constexpr (OUT == TK3D_MLP_OUT_MASK) {
                const f32x4 was = *reinterpret_cast<const f32x4 *>(p.yprev + offset);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v[k] = (inside & passes(normalised(was[k], norm))) ? v[k] : 0.0f;
                    s1 += v[k];
                    s2 = __builtin_fmaf(v[k], was[k] - norm.x, s2);
                }
            }
            float *out = p.out;
            int64_t to = offset;
            if constexpr (OUT == TK3D_MLP_OUT_PLAIN) {
                const bool one = c < p.C0;
                out = one ? p.out : p.out2;
                to = ((int64_t)b * (one ? p.C0 : C - p.C0) + (one ? c : c - p.C0)) * P + pos;
            }
            if (out && channel < C && inside)
                *reinterpret_cast<f32x4 *>(out + to) = v;
        }
        sum1[j] = s1;
        sum2[j] = s2;
    }
    if constexpr (OUT == TK3D_MLP_OUT_MASK) {
        __syncthreads();
        double2 *part = reinterpret_cast<double2 *>(lds);  // [wave][32 CT]
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            sum1[j] += __shfl_xor(sum1[j], 32);
            sum2[j] += __shfl_xor(sum2[j], 32);
            if (half == 0)
                part[wave * (32 * CT) + j * 32 + l32] = double2{sum1[j], sum2[j]};
        }
        __syncthreads();
        if (tid < 32 * CT && cbase + tid < C) {
            double2 v = part[tid];
            for (int i = 1; i < kWideWaves; ++i) {
                v.x += part[i * (32 * CT) + tid].x;
                v.y += part[i * (32 * CT) + tid].y;
            }
            reinterpret_cast<double2 *>(p.partial)[(int64_t)(cbase + tid) * a.groups + group] = v;
        }
    }
}

// ---- launches ----------------------------------------------------------------------------------------------

bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int ROW, int COL> int launch_outer(const WideOuterArgs &a, hipStream_t stream)
{
    mlp_wide_outer_kernel<ROW, COL><<<placed(a.splits * a.rblocks, a.cblocks), kWide, 0, stream>>>(a);
    return tk_launch_status();
}

template <int IN, int OUT, int CT> int launch_product(const WideProductArgs &a, hipStream_t stream)
{
    const int tables = a.chunks * 32 * 16 * (IN == TK3D_MLP_IN_GRAD_OUT ? 2 : 1);
    int bytes = 2 * 32 * (kWidePositions + 4 + 32 * CT + 4) * 4 + tables;
    constexpr int sums = kWideWaves * 4096;  // (also more than the partial sums of 160 channels)
    bytes = bytes > sums ? bytes : sums;
    if (bytes > 160 << 10)
        return TK3D_ERR_UNSUPPORTED;
    const int rc = tk_allow_dynamic_lds<mlp_wide_product_kernel<IN, OUT, CT>>(160 << 10);
    if (rc != TK3D_OK)
        return rc;
    mlp_wide_product_kernel<IN, OUT, CT><<<placed(a.groups, a.cblocks), kWide, bytes, stream>>>(a);
    return tk_launch_status();
}

struct ProductShape {
    int ct, groups, tiles, cblocks;
};

// Where three of four CUs get a workgroup; with fewer mlp_split_kernel is as fast or faster (256 -> 384
// channels, 4096 positions: four teams and 64 positions a workgroup 17.9, split 15.9 us).
ProductShape product_shape(int in, int out, const tk3d_mlp_product &p)
{
    const ProductShape none{0, 0, 0, 0};
    const tk3d_mlp_source &s = p.src[0];
    const bool grad = in == TK3D_MLP_IN_GRAD || in == TK3D_MLP_IN_GRAD_OUT;
    if ((!grad && in != TK3D_MLP_IN_CENTRED && in != TK3D_MLP_IN_SHIFTED) ||
        (out != TK3D_MLP_OUT_MASK && out != TK3D_MLP_OUT_PLAIN) || s.K <= 64 || s.K > 2048 || p.C <= 64 ||
        p.P % 4 != 0 || !aligned(s.x) || (grad && !aligned(s.y)) || s.batch_stride % 4 != 0 ||
        !aligned(p.out) || !aligned(p.out2) || !aligned(p.yprev) || !aligned(p.add))
        return none;
    const int ctiles = (p.C + 31) / 32;
    const int ct = ctiles % 5 == 0 ? 5 : ctiles % 4 == 0 ? 4 : ctiles % 3 == 0 ? 3 : 4;
    const int cblocks = (ctiles + ct - 1) / ct, tiles = (p.P + kWidePositions - 1) / kWidePositions;
    if ((int64_t)p.B * tiles * cblocks < tk_cu_count() * 3 / 4 || (int64_t)p.B * tiles * cblocks > (1 << 24))
        return none;
    return {ct, p.B * tiles, tiles, cblocks};
}

}  // namespace

// Rows and columns are the same activations, less the same centres: half of the blocks leave at once. (For the
// number of splits alone.)
static bool symmetric(const tk3d_mlp_outer &p) { return p.row.x == p.col.x && p.row.y == nullptr && p.row.K == p.col.K; }

// Rows of one or two tiles of 32, and columns of one, waste too much of 128 x 64. No fewer positions than
// a tile for a workgroup, else two workgroups to a CU.
int tk_mlp_wide_outer_splits(const tk3d_mlp_outer &p)
{
    if (p.row.K <= 64 || p.col.K <= 32 || p.P % 4 != 0 || !aligned(p.row.x) || !aligned(p.row.y) || !aligned(p.col.x) ||
        p.row.batch_stride % 4 != 0 || p.col.batch_stride % 4 != 0)
        return 0;
    const int64_t rblocks = (p.row.K + 127) / 128, cblocks = (p.col.K + 63) / 64;
    int64_t blocks = rblocks * cblocks;
    if (symmetric(p))  // blocks on and above the diagonal: cblocks - 2 r of row block r
        blocks -= rblocks * (rblocks - 1);
    const int64_t total = (int64_t)p.B * ((p.P + 31) / 32);
    if (total > (1 << 29) || blocks > (1 << 20))
        return 0;
    int64_t splits = 2 * tk_cu_count() / blocks;
    splits = splits > total ? total : splits;
    return splits < 1 ? 1 : (int)splits;
}

int tk_mlp_wide_outer(int row, int col, const tk3d_mlp_outer &p, hipStream_t stream)
{
    WideOuterArgs a;
    a.p = p;
    a.tiles = (p.P + 31) / 32;
    a.total = p.B * a.tiles;
    a.splits = tk_mlp_wide_outer_splits(p);
    a.rblocks = (p.row.K + 127) / 128;
    a.cblocks = (p.col.K + 63) / 64;
#define TK_CASE(ROW, COL)                                                                       \
    if (row == ROW && col == COL)                                                               \
        return launch_outer<ROW, COL>(a, stream);
    TK_CASE(TK3D_MLP_ROW_RAW, TK3D_MLP_COL_RAW)
    TK_CASE(TK3D_MLP_ROW_GRAD, TK3D_MLP_COL_RAW)
    TK_CASE(TK3D_MLP_ROW_GRAD, TK3D_MLP_COL_ACT)
    TK_CASE(TK3D_MLP_ROW_GRAD_OUT, TK3D_MLP_COL_RAW)
    TK_CASE(TK3D_MLP_ROW_GRAD_OUT, TK3D_MLP_COL_ACT)
    TK_CASE(TK3D_MLP_ROW_CENTRED, TK3D_MLP_COL_CENTRED)
    TK_CASE(TK3D_MLP_ROW_SHIFTED, TK3D_MLP_COL_SHIFTED)
#undef TK_CASE
    return TK3D_ERR_UNSUPPORTED;
}

int tk_mlp_wide_product_slots(int in, int out, const tk3d_mlp_product &p) { return product_shape(in, out, p).groups; }

int tk_mlp_wide_product(int in, int out, const tk3d_mlp_product &p, hipStream_t stream)
{
    const ProductShape s = product_shape(in, out, p);
    WideProductArgs a{p, s.tiles, s.groups, s.cblocks, (p.src[0].K + 31) / 32, 0};
    a.rows4 = p.src[0].wc == 1 && p.src[0].wk % 4 == 0 && p.C % 4 == 0 && aligned(p.src[0].w);
#define TK_SHAPE(IN, OUT, CT)                                                                   \
    if (s.ct == CT)                                                                             \
        return launch_product<IN, OUT, CT>(a, stream);
#define TK_CASE(IN, OUT)                                                                        \
    if (in == IN && out == OUT) {                                                               \
        TK_SHAPE(IN, OUT, 3)                                                                    \
        TK_SHAPE(IN, OUT, 4)                                                                    \
        TK_SHAPE(IN, OUT, 5)                                                                    \
    }
    TK_CASE(TK3D_MLP_IN_GRAD, TK3D_MLP_OUT_MASK)
    TK_CASE(TK3D_MLP_IN_GRAD, TK3D_MLP_OUT_PLAIN)
    TK_CASE(TK3D_MLP_IN_GRAD_OUT, TK3D_MLP_OUT_MASK)
    TK_CASE(TK3D_MLP_IN_GRAD_OUT, TK3D_MLP_OUT_PLAIN)
    TK_CASE(TK3D_MLP_IN_CENTRED, TK3D_MLP_OUT_MASK)
    TK_CASE(TK3D_MLP_IN_SHIFTED, TK3D_MLP_OUT_PLAIN)
#undef TK_CASE
#undef TK_SHAPE
    return TK3D_ERR_UNSUPPORTED;
}
