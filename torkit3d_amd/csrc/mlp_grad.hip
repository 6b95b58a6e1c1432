// Backward of a shared-MLP layer in one pass: the gradient of its input and that of its weights read the
// same tensors (include/tk3d_mlp.h, tk3d_mlp_pair_f32).
//
// What bounds it: apart, mlp_product_kernel and mlp_outer_kernel (mlp.hip) read the gradient, y and the
// input twice, seven tensors moved where four do, and a load of the outer product, whose lanes read runs of a
// row each, touches 64 cache lines. Together the floors of memory and of the fp32 matrix rate are 57 and 56 us
// for 128 -> 128 channels and 131072 positions; on fewer channels memory's is the higher one.
//
// A workgroup of eight waves has a CU to itself and walks over tiles of positions. The tile's gradient and
// activations, normalised on the way, lie in LDS; while one tile is multiplied the next is on its way from
// memory in registers and is then written to the other half of LDS, one barrier a tile. Waves 0 to 3 form
// W^T dy, their weights in registers for the whole launch; waves 4 to 7 form dy x^T, in registers too: every
// SIMD has a wave of either kind with the same number of matrix instructions.
//
// us, apart -> together (masked gradient | centred activations):
//   128 -> 128 channels, 131072 positions 152 -> 95 | 140 -> 82;  16384 positions 31 -> 19 | 29 -> 19
//   64 -> 64, 262144 positions 123 -> 59 | 96 -> 58;  2048 positions 17.6 -> 7.2 | 16.4 -> 7.5
//   32 -> 32, 524288 positions 91 -> 50 | 72 -> 44;  128 -> 64, 131072 positions 99 -> 51
// At 128 channels what is left over the floors is the part of a tile in which waves 0 to 3 mask and store
// and the matrix cores have the other waves' work alone; a launch of one tile a CU takes 10 us, for weights,
// partial sums and the first tile's trip. Errors against 64 bits are those of the separate kernels or less
// (dx 2.1e-7 -> 1.1e-7, dW 2.9e-7 -> 1.3e-7 of the result at 128 channels): chains are shorter.
#include "mlp_common.h"

namespace {

constexpr int kPairBlock = 512, kHalf = kPairBlock / TK_WAVE / 2, kLoaders = kPairBlock / 2;

enum PairIn { GRAD, GRAD_OUT, CENTRED };  // as TK3D_MLP_ROW_*
enum PairOut { MASK, PLAIN };

struct PairArgs {
    tk3d_mlp_product p;
    tk3d_mlp_outer o;
    int tiles, total;  // tiles of positions: per batch element, in all
};

// OT and IT: tiles of 32 output and input channels of the layer.
template <int IN, int OUT, int OT, int IT> struct Pair {
    static constexpr int NPT = 4 / IT, NP = 32 * NPT;  // positions of a tile, so that dx has a 32 x 32 tile a wave
    static constexpr int QUADS = NP / 4, ROWS = kLoaders / QUADS;
    static constexpr int STRIDE = NP + 4;  // of a row in LDS: reads of 16 bytes by rows hit all banks
    static constexpr int DEPTH = IN == CENTRED ? IT : OT;  // tiles of 32 that dx adds up
    static constexpr int GL = IN == CENTRED ? 0 : 32 * OT / ROWS, XL = 32 * IT / ROWS;  // 16-byte loads a thread
    static constexpr int G = IN == CENTRED ? 0 : 32 * OT * STRIDE, X = 32 * IT * STRIDE;
    static constexpr int HALF = G + X + (OUT == MASK ? X : 0);
    static constexpr int TABLE = 4 * ((IN == CENTRED ? 0 : 32 * OT) + (IN == GRAD_OUT ? 32 * OT : 0) +
                                      (OUT == MASK ? 32 * IT : 0));
    static constexpr int BYTES = 4 * (TABLE + 2 * HALF);
    // dW: tiles of a wave, and waves that share a tile's positions
    static constexpr int T = OT * IT;
    static constexpr int RT = T == 16 || (T == 8 && IT == 4) ? 2 : 1;
    static constexpr int CT = T == 16 || (T == 8 && IT == 2) ? 2 : 1;
    static constexpr int SP = T < kHalf ? kHalf / T : 1;
    static_assert(IN != CENTRED || OT == IT, "rows and columns are the same");
    static_assert(GL * ROWS == (IN == CENTRED ? 0 : 32 * OT) && XL * ROWS == 32 * IT, "whole loads");
    static_assert(kHalf * RT * CT == T * SP, "every tile once");
    static_assert(BYTES <= 160 << 10, "LDS of a CU");
};

__device__ __forceinline__ f32x4 read(const float *base, unsigned offset)
{
    return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(base) + offset);
}

template <int IN, int OUT, int OT, int IT>
__global__ void __launch_bounds__(kPairBlock) mlp_pair_kernel(PairArgs a)
{
    typedef Pair<IN, OUT, OT, IT> S;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const tk3d_mlp_product &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, l32 = lane & 31;
    const int P = p.P, R = a.o.row.K, I = p.C;

    f32x4 *grad_coef = reinterpret_cast<f32x4 *>(lds);
    f32x4 *grad_act = grad_coef + (IN == CENTRED ? 0 : 32 * OT);
    f32x4 *x_act = grad_act + (IN == GRAD_OUT ? 32 * OT : 0);
    float *halves = lds + S::TABLE;
    if constexpr (IN != CENTRED)
        for (int r = tid; r < 32 * OT; r += kPairBlock) {
            const int row = r < R ? r : R - 1;
            grad_coef[r] = reinterpret_cast<const f32x4 *>(p.src[0].coef)[row];
            if constexpr (IN == GRAD_OUT)
                grad_act[r] = constants_of(p.in_norm, row);
        }
    if constexpr (OUT == MASK)
        for (int r = tid; r < 32 * IT; r += kPairBlock)
            x_act[r] = constants_of(p.out_norm, r < I ? r : I - 1);
    __syncthreads();

    // A thread's 16 bytes of every S::ROWS-th row of a tile: waves 4 to 7 bring the gradient, waves 0 to 3 the
    // input (if both came with one kind of wave, that was the kind the others waited for: 128 -> 128 channels,
    // 131072 positions 100 us). The rows' constants stay in registers.
    const int quad = tid % kLoaders % S::QUADS, row0 = tid % kLoaders / S::QUADS;
    const auto place = [&](int tile, int &b, int &at) {
        b = tile / a.tiles;
        const int pos = (tile - b * a.tiles) * S::NP + 4 * quad;
        at = pos < P ? pos : P - 4;
        return pos < P;
    };
    const auto row_of = [&](int r, int rows, int at) {  // (32-bit byte offsets, see pair_shape)
        return ((unsigned)(r < rows ? r : rows - 1) * (unsigned)P + (unsigned)at) * 4u;
    };
    // Rows and positions past the last ones are zero, so that nothing comes of them.
    struct Gradients {
        f32x4 e[S::GL ? S::GL : 1], y[S::GL ? S::GL : 1], coef[S::GL ? S::GL : 1];
    } gradients;
    const auto load_gradients = [&](int tile) {
        int b, at;
        place(tile, b, at);
        const int64_t batch = (int64_t)b * p.src[0].batch_stride;
#pragma unroll
        for (int i = 0; i < S::GL; ++i) {
            const unsigned offset = row_of(row0 + i * S::ROWS, R, at);
            gradients.e[i] = read(p.src[0].x + batch, offset);
            gradients.y[i] = read(p.src[0].y + batch, offset);
        }
    };
    const auto store_gradients = [&](int tile, float *to) {
        int b, at;
        const bool in = place(tile, b, at);
        to += row0 * S::STRIDE + 4 * quad;
#pragma unroll
        for (int i = 0; i < S::GL; ++i) {
            const int r = row0 + i * S::ROWS;
            const f32x4 k = gradients.coef[i], y = gradients.y[i];
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float g = gradients.e[i][j];
                if constexpr (IN == GRAD_OUT)
                    g = passes(normalised(y[j], grad_act[r])) ? g : 0.0f;
                g = __builtin_fmaf(k.x, g, __builtin_fmaf(k.y, y[j], k.z));
                v[j] = in && r < R ? g : 0.0f;
            }
            *reinterpret_cast<f32x4 *>(to + i * S::ROWS * S::STRIDE) = v;
        }
    };
    struct Inputs {
        f32x4 x[S::XL], act[S::XL];
    } inputs;
    const auto load_inputs = [&](int tile) {
        int b, at;
        place(tile, b, at);
#pragma unroll
        for (int i = 0; i < S::XL; ++i)
            inputs.x[i] = read(a.o.col.x + (int64_t)b * a.o.col.batch_stride, row_of(row0 + i * S::ROWS, I, at));
    };
    const auto store_inputs = [&](int tile, float *to) {
        int b, at;
        const bool in = place(tile, b, at);
        to += S::G + row0 * S::STRIDE + 4 * quad;
#pragma unroll
        for (int i = 0; i < S::XL; ++i) {
            float *row = to + i * S::ROWS * S::STRIDE;
            f32x4 v = inputs.x[i];
            if constexpr (OUT == MASK) {
                *reinterpret_cast<f32x4 *>(row + S::X) = v;
                const f32x4 k = inputs.act[i];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = relu(normalised(v[j], k));
                    if constexpr (IN == CENTRED)
                        v[j] -= centre_of(k);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = in && row0 + i * S::ROWS < I ? v[j] : 0.0f;
            *reinterpret_cast<f32x4 *>(row) = v;
        }
    };
    const auto input_constants = [&] {
#pragma unroll
        for (int i = 0; i < S::XL; ++i)
            if constexpr (OUT == MASK)
                inputs.act[i] = x_act[row0 + i * S::ROWS];
    };

    const bool forms_dx = wave < kHalf;
    // dx: a wave's 32 channels and its 32 positions of a tile.
    const int dx_channels = (wave % IT) * 32, dx_positions = (wave / IT) % S::NPT * 32;
    const int channel = dx_channels + l32, c = channel < I ? channel : I - 1;
    // dW: a wave's tiles, and its share of the positions.
    const int share = wave - kHalf;
    const int tile0 = S::T == 16 ? (share >> 1) * 2 * IT + (share & 1) * 2
                      : S::T == 8 ? (IT == 2 ? share * IT : share) : share % S::T;
    const int dw_rows = tile0 / IT * 32, dw_columns = tile0 % IT * 32;
    const int dw_from = S::T < kHalf ? share / S::T * (S::NP / S::SP) : 0;

    float w[16 * S::DEPTH];
    double sum1 = 0.0, sum2 = 0.0;
    f32x4 constants{0.0f, 0.0f, 0.0f, 0.0f};
    float bias = 0.0f;
    f32x4 out[4];
    const auto form_dx = [&](int tile, const float *from) {
        const int b = tile / a.tiles, pos0 = (tile - b * a.tiles) * S::NP + dx_positions + 4 * half;
        const int64_t row = ((int64_t)b * I + c) * P;
        f32x4 add[4];
        if constexpr (IN == CENTRED)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                add[q] = *reinterpret_cast<const f32x4 *>(p.add + row + (pos0 + 8 * q < P ? pos0 + 8 * q : P - 4));
        // Two chains side by side, so that one always has a step ready, of up to 32 channels each, and the
        // next four reads on their way while four steps are multiplied.
        constexpr int LENGTH = S::DEPTH > 1 ? 16 : 8, GROUPS = 16 * S::DEPTH / 4;
        tk_f32x16 sum, acc[2];
        float v[2][4];
        const float *in = from + half * S::STRIDE + dx_positions + l32;
        const auto step_of = [](int group, int i) {  // the i-th of a group: even i in one chain, odd in the other
            const int in_chain = 2 * group % LENGTH + i / 2;
            return 2 * group / LENGTH * 2 * LENGTH + (i & 1) * LENGTH + in_chain;
        };
        const auto fetch = [&](int group) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[group & 1][i] = in[2 * step_of(group, i) * S::STRIDE];
        };
        fetch(0);
#pragma unroll
        for (int group = 0; group < GROUPS; ++group) {
            if (group + 1 < GROUPS)
                fetch(group + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (2 * group % LENGTH == 0)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[0][r] = acc[1][r] = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[group & 1][i], w[step_of(group, i)], acc[i & 1],
                                                                  0, 0, 0);
            if (2 * (group + 1) % LENGTH == 0)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    sum[r] = 2 * (group + 1) == LENGTH ? acc[0][r] + acc[1][r] : sum[r] + (acc[0][r] + acc[1][r]);
        }
        const float *before = from + S::G + S::X + channel * S::STRIDE + dx_positions + 4 * half;
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x4 was;
            if constexpr (OUT == MASK)
                was = *reinterpret_cast<const f32x4 *>(before + 8 * q);
            const bool inside = pos0 + 8 * q < P;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                out[q][j] = sum[4 * q + j] + bias;
                if constexpr (IN == CENTRED)
                    out[q][j] += add[q][j];
                if constexpr (OUT == MASK) {
                    // (no branch: `&`)
                    out[q][j] = (inside & passes(normalised(was[j], constants))) ? out[q][j] : 0.0f;
                    s1 += out[q][j];
                    s2 = __builtin_fmaf(out[q][j], was[j] - constants.x, s2);
                }
            }
        }
        sum1 += (double)s1;
        sum2 += (double)s2;
    };
    const auto put = [&](int tile) {
        const int b = tile / a.tiles, pos0 = (tile - b * a.tiles) * S::NP + dx_positions + 4 * half;
        float *row = p.out + ((int64_t)b * I + c) * P;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (channel < I && pos0 + 8 * q < P)
                *reinterpret_cast<f32x4 *>(row + pos0 + 8 * q) = out[q];
    };

    // Sums of a tile (16 to 32 steps of the product) on top of those of the tiles before it: chains are
    // shorter than in mlp_outer_kernel.
    tk_f32x16 total[S::RT][S::CT];
    double row_total[S::RT];
#pragma unroll
    for (int i = 0; i < S::RT; ++i) {
        row_total[i] = 0.0;
#pragma unroll
        for (int j = 0; j < S::CT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                total[i][j][r] = 0.0f;
    }
    const auto form_dw = [&](const float *from) {
        tk_f32x16 acc[S::RT][S::CT];
#pragma unroll
        for (int i = 0; i < S::RT; ++i)
#pragma unroll
            for (int j = 0; j < S::CT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[i][j][r] = 0.0f;
        const int at = dw_from + 4 * half;
        const float *rows = from + (dw_rows + l32) * S::STRIDE + at;
        const float *columns = from + S::G + (dw_columns + l32) * S::STRIDE + at;
        float row_sum[S::RT] = {};
        f32x4 g[2][S::RT], h[2][S::CT];
        const auto fetch = [&](int step) {
#pragma unroll
            for (int i = 0; i < S::RT; ++i)
                g[step & 1][i] = *reinterpret_cast<const f32x4 *>(rows + i * 32 * S::STRIDE + 8 * step);
#pragma unroll
            for (int j = 0; j < S::CT; ++j)
                h[step & 1][j] = *reinterpret_cast<const f32x4 *>(columns + j * 32 * S::STRIDE + 8 * step);
        };
        constexpr int STEPS = S::NP / S::SP / 8;
        fetch(0);
#pragma unroll
        for (int step = 0; step < STEPS; ++step) {
            if (step + 1 < STEPS)
                fetch(step + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < S::RT; ++i) {
                    if constexpr (IN == CENTRED)
                        row_sum[i] += g[step & 1][i][k];
#pragma unroll
                    for (int j = 0; j < S::CT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(g[step & 1][i][k], h[step & 1][j][k],
                                                                        acc[i][j], 0, 0, 0);
                }
        }
#pragma unroll
        for (int i = 0; i < S::RT; ++i) {
            row_total[i] += (double)row_sum[i];
#pragma unroll
            for (int j = 0; j < S::CT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    total[i][j][r] += acc[i][j][r];
        }
    };

    // Each kind of wave has a loop of its own, with the same barriers.
    const int step = gridDim.x;  // (no more than there are tiles)
    if (forms_dx) {
        const int K = p.src[0].K;
#pragma unroll
        for (int s = 0; s < 16 * S::DEPTH; ++s) {
            const int k = 2 * s + half;
            w[s] = p.src[0].w[(int64_t)(k < K ? k : K - 1) * p.src[0].wk + (int64_t)c * p.src[0].wc];
        }
#pragma unroll
        for (int s = 0; s < 16 * S::DEPTH; ++s)
            w[s] = 2 * s + half < K && channel < I ? w[s] : 0.0f;
        if constexpr (OUT == MASK)
            constants = x_act[channel];
        if (p.bias)
            bias = p.bias[c];
        // (behind the weights: with these at hand nothing else is waited for in the loop)
        if constexpr (IN != CENTRED) {
            input_constants();
            load_inputs(blockIdx.x);
            store_inputs(blockIdx.x, halves);
        }
        __syncthreads();
        for (int tile = blockIdx.x, now = 0; tile < a.total; tile += step, now ^= 1) {
            const bool more = IN != CENTRED && tile + step < a.total;
            if (more)
                load_inputs(tile + step);
            form_dx(tile, halves + now * S::HALF);
            if (more)
                store_inputs(tile + step, halves + (now ^ 1) * S::HALF);
            put(tile);  // (not before: what was loaded would be waited for behind it)
            __syncthreads();
        }
    } else {
        const auto load = [&](int tile) {
            if constexpr (IN == CENTRED)
                load_inputs(tile);
            else
                load_gradients(tile);
        };
        const auto store = [&](int tile, float *to) {
            if constexpr (IN == CENTRED)
                store_inputs(tile, to);
            else
                store_gradients(tile, to);
        };
        if constexpr (IN == CENTRED)
            input_constants();
#pragma unroll
        for (int i = 0; i < S::GL; ++i)
            gradients.coef[i] = grad_coef[row0 + i * S::ROWS];
        load(blockIdx.x);
        store(blockIdx.x, halves);
        __syncthreads();
        for (int tile = blockIdx.x, now = 0; tile < a.total; tile += step, now ^= 1) {
            if (tile + step < a.total)
                load(tile + step);
            form_dw(halves + now * S::HALF);
            if (tile + step < a.total)
                store(tile + step, halves + (now ^ 1) * S::HALF);
            __syncthreads();
        }
    }

    // (everything below is behind the loop's last barrier)
    constexpr int TILE = 16 * TK_WAVE;
    double2 *sums = reinterpret_cast<double2 *>(lds);              // [kHalf][32]
    double *row_sums = reinterpret_cast<double *>(sums + kHalf * 32);  // [kHalf][RT * 32]
    float *shares = reinterpret_cast<float *>(row_sums + kHalf * S::RT * 32);  // [kHalf][TILE]
    if (forms_dx) {
        sum1 += __shfl_xor(sum1, 32);
        sum2 += __shfl_xor(sum2, 32);
        if (half == 0)
            sums[wave * 32 + l32] = double2{sum1, sum2};
    } else {
#pragma unroll
        for (int i = 0; i < S::RT; ++i) {
            row_total[i] += __shfl_xor(row_total[i], 32);
            if (half == 0)
                row_sums[(share * S::RT + i) * 32 + l32] = row_total[i];
#pragma unroll
            for (int j = 0; j < S::CT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = dw_rows + i * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
                    const int column = dw_columns + j * 32 + l32;
                    if (S::SP > 1)
                        shares[share * TILE + r * TK_WAVE + lane] = total[i][j][r];
                    else if (row < R && column < I)
                        a.o.partial[((int64_t)blockIdx.x * R + row) * I + column] = total[i][j][r];
                }
        }
    }
    __syncthreads();
    if constexpr (S::SP > 1)
        for (int at = tid; at < S::T * TILE; at += kPairBlock) {
            const int t = at / TILE, r = at % TILE / TK_WAVE, l = at % TK_WAVE;
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < S::SP; ++k)
                s += shares[(k * S::T + t) * TILE + at % TILE];
            const int row = t / IT * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), column = t % IT * 32 + (l & 31);
            if (row < R && column < I)
                a.o.partial[((int64_t)blockIdx.x * R + row) * I + column] = s;
        }
    if constexpr (OUT == MASK)
        if (tid < I) {
            double2 s{0.0, 0.0};
#pragma unroll
            for (int k = 0; k < S::NPT; ++k) {
                s.x += sums[(k * IT + tid / 32) * 32 + tid % 32].x;
                s.y += sums[(k * IT + tid / 32) * 32 + tid % 32].y;
            }
            reinterpret_cast<double2 *>(p.partial)[(int64_t)tid * gridDim.x + blockIdx.x] = s;
        }
    if constexpr (IN == CENTRED)
        if (a.o.rowsum && tid < R) {  // rows of tile t: the waves of the tiles (t, 0)
            const int t = tid / 32;
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < S::SP; ++k) {
                const int owner = S::T == 16 ? t / 2 * 2 : S::T == 4 ? t * IT : k * S::T;
                s += row_sums[(owner * S::RT + (S::T == 16 ? t % 2 : 0)) * 32 + tid % 32];
            }
            a.o.rowsum[(int64_t)blockIdx.x * R + tid] = (float)s;
        }
}

template <int IN, int OUT, int OT, int IT> int launch_pair(PairArgs &a, int grid, hipStream_t stream)
{
    typedef Pair<IN, OUT, OT, IT> S;
    const int rc = tk_allow_dynamic_lds<mlp_pair_kernel<IN, OUT, OT, IT>>(S::BYTES);
    if (rc != TK3D_OK)
        return rc;
    mlp_pair_kernel<IN, OUT, OT, IT><<<grid, kPairBlock, S::BYTES, stream>>>(a);
    return tk_launch_status();
}

struct PairShape {
    int ot, it, grid, tiles, total;
};

// The tiles of a layer, or {0}: up to 128 channels on either side, except 128 from 32, whose gradient does
// not fit in LDS twice, 16-byte rows, and 32-bit byte offsets within a batch element. At any number of positions:
// 128 -> 128 channels, 2048 positions 18.9 apart, 12.2 us together.
bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
PairShape pair_shape(const tk3d_mlp_product &p, const tk3d_mlp_outer &o)
{
    const int O = o.row.K, I = p.C;
    PairShape s{0, 0, 0, 0, 0};
    if (O > 128 || I > 128 || p.P % 4 != 0 || p.B <= 0 || p.P <= 0 ||
        !tk_fits(1 << 29, (O > I ? O : I) + 8, p.P) ||
        !aligned(p.src[0].x) || !aligned(p.src[0].y) || !aligned(p.out) || !aligned(p.yprev) || !aligned(p.add) ||
        !aligned(o.col.x) || p.src[0].batch_stride % 4 != 0 || o.col.batch_stride % 4 != 0)
        return s;
    const auto tiles_of = [](int c) { return c > 64 ? 4 : c > 32 ? 2 : 1; };
    const int it = tiles_of(I);
    const int ot = tiles_of(O);
    if (ot == 4 && it == 1)
        return s;
    const int np = 32 * (4 / it);
    const int64_t tiles = (p.P + np - 1) / np, total = tiles * p.B;
    const int64_t most = tk_cu_count();
    if (total > TK_MAX_I32 - 2 * most)  // (a workgroup looks two of its tiles ahead)
        return s;
    return {ot, it, (int)(total < most ? total : most), (int)tiles, (int)total};
}

}  // namespace

extern "C" {

int tk3d_mlp_pair_slots(const tk3d_mlp_product *p, const tk3d_mlp_outer *o)
{
    return pair_shape(*p, *o).grid;
}

int tk3d_mlp_pair_f32(int in, int out, const tk3d_mlp_product *p, const tk3d_mlp_outer *o, void *stream_)
{
    if (!p || !o)
        return TK3D_ERR_NULL_POINTER;
    const PairShape s = pair_shape(*p, *o);
    if (s.grid == 0 || p->B != o->B || p->P != o->P || p->C != o->col.K || p->src[0].K != o->row.K)
        return TK3D_ERR_UNSUPPORTED;
    PairArgs a{*p, *o, s.tiles, s.total};
    const hipStream_t stream = (hipStream_t)stream_;
#define TK_SHAPE(IN, OUT, OT, IT)                                                               \
    if (s.ot == OT && s.it == IT)                                                               \
        return launch_pair<IN, OUT, OT, IT>(a, s.grid, stream);
#define TK_CASE(IN, OUT)                                                                        \
    if (in == TK3D_MLP_IN_##IN && out == TK3D_MLP_OUT_##OUT) {                                  \
        TK_SHAPE(IN, OUT, 1, 1)                                                                 \
        TK_SHAPE(IN, OUT, 2, 2)                                                                 \
        TK_SHAPE(IN, OUT, 4, 4)                                                                 \
        if constexpr (IN != CENTRED) {                                                          \
            TK_SHAPE(IN == CENTRED ? GRAD : IN, OUT, 1, 2)                                      \
            TK_SHAPE(IN == CENTRED ? GRAD : IN, OUT, 2, 1)                                      \
            TK_SHAPE(IN == CENTRED ? GRAD : IN, OUT, 1, 4)                                      \
            TK_SHAPE(IN == CENTRED ? GRAD : IN, OUT, 2, 4)                                      \
            TK_SHAPE(IN == CENTRED ? GRAD : IN, OUT, 4, 2)                                      \
        }                                                                                       \
    }
    TK_CASE(GRAD, MASK)
    TK_CASE(GRAD_OUT, MASK)
    TK_CASE(CENTRED, MASK)
    TK_CASE(GRAD, PLAIN)
    TK_CASE(GRAD_OUT, PLAIN)
#undef TK_CASE
#undef TK_SHAPE
    return TK3D_ERR_UNSUPPORTED;
}

}  // extern "C"
