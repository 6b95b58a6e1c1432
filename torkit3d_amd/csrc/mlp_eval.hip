// A shared MLP of three layers between a grouping and the maximum over its neighbours, in evaluation
// (include/tk3d_mlp.h, tk3d_mlp_grouped_pool_f32): one launch in place of one a layer, and the activations
// between the layers stay in LDS.
//
// A workgroup takes 64 grouped positions at a time: two groups of 32 or one of 64.
//   1. The first layer as in mlp_group_kernel: a lane is a position, gathers its point's row of the product
//      with the features, adds the centred coordinates' part and leaves its activations in LDS, four channels
//      of a position side by side.
//   2. The second layer on the matrix cores: rows of the instruction are channels, columns positions, so that
//      a lane's results are four channels of a position again, 16 bytes of LDS.
//   3. The third with rows and columns exchanged: a lane's results are 16 positions of one channel, whose
//      maximum is taken in registers. Only maxima go to memory.
// Both operands are read as 16 bytes a lane and group of eight channels (half a wave's lanes have the first
// four, half the others; the order within a sum is the kernels' own): the activations from LDS, rows padded by 16
// bytes, without bank conflicts, the weights from L2 straight into registers, 16 channels ahead. Sums are in
// fp32 and in chains of 16 channels, as evaluation's other products are.
//
// What bounds it: one cloud is latency (one layer's LDS and weights behind the other's), large batches are the
// matrix rate. Three launches and this one, with the features' product, us: 1 x 512 groups of 32, 64-64-128 channels
// 19.6, 12.9 (which is host time); 1 x 128 groups of 64, 128-128-256 29.3, 22.1; 32 x 512 groups of 32 203, 142;
// 32 x 128 groups of 64 332, 262 (103 TFLOP/s in this launch); 8 x 2048 groups of 32, 32-32-64 95, 67.
#include "mlp_common.h"

namespace {

struct GroupedArgs {
    tk3d_mlp_grouped_pool p;
    int tiles;  // per batch element
    int total;
    int part;   // output channels of a workgroup, a multiple of 32
};

// A lane's weights of a block of 16 * D channels: at `w` its output channel's row at its half's channels.
template <int D> struct Weights {
    f32x4 v[2 * D];
    __device__ __forceinline__ void load(const float *w)
    {
#pragma unroll
        for (int g = 0; g < 2 * D; ++g)
            v[g] = *reinterpret_cast<const f32x4 *>(w + 8 * g);
    }
};

// sum over the K (a multiple of 16 D) activations of PT times 32 positions times a row of weights, the first
// block of which is `now`. `x` is the lane's position at its half's LDS row, ROW the rows' length.
template <int PT, int D, int ROW, bool CHANNEL_ROWS>
__device__ __forceinline__ void product(const f32x4 *x, Weights<D> &now, const float *w, int K,
                                        tk_f32x16 (&total)[PT])
{
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            total[t][i] = 0.0f;
    for (int k = 0; k < K; k += 16 * D) {
        Weights<D> next;
        if (k + 16 * D < K)
            next.load(w + k + 16 * D);
#pragma unroll
        for (int d = 0; d < D; ++d) {  // a chain
            f32x4 v[2][PT];
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int t = 0; t < PT; ++t)
                    v[g][t] = x[(k / 4 + 4 * d + 2 * g) * ROW + 32 * t];
            tk_f32x16 acc[PT];
#pragma unroll
            for (int t = 0; t < PT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    acc[t][i] = 0.0f;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int t = 0; t < PT; ++t) {
                        const float in = v[g][t][q], weight = now.v[2 * d + g][q];
                        acc[t] = CHANNEL_ROWS ? __builtin_amdgcn_mfma_f32_32x32x2f32(weight, in, acc[t], 0, 0, 0)
                                              : __builtin_amdgcn_mfma_f32_32x32x2f32(in, weight, acc[t], 0, 0, 0);
                    }
#pragma unroll
            for (int t = 0; t < PT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    total[t][i] += acc[t][i];
        }
        now = next;
    }
}

// NW waves, tiles of TP positions.
template <int NW, int TP>
__global__ void __launch_bounds__(NW *TK_WAVE, 4) mlp_grouped_pool_kernel(GroupedArgs a)
{
    constexpr int ROW = TP + 1;  // LDS row of four channels, in 16-byte words
    constexpr int PT = TP / 32, D = PT == 1 ? 2 : 1;
    extern __shared__ f32x4 lds[];
    const tk3d_mlp_grouped_pool &p = a.p;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int C1 = p.C[0], C2 = p.C[1], C3 = p.C[2];
    const int P = p.M * p.S;
    const int cbase = blockIdx.y * a.part;
    const int channels = C3 - cbase < a.part ? C3 - cbase : a.part;
    f32x4 *act1 = lds, *act2 = act1 + C1 / 4 * ROW;
    f32x4 *norm1 = act2 + C2 / 4 * ROW, *norm2 = norm1 + C1, *norm3 = norm2 + C2, *wx = norm3 + a.part;
    for (int c = tid; c < C1; c += NW * TK_WAVE) {
        norm1[c] = constants_of(p.norm[0], c);
        const float *w = p.wx + (int64_t)c * p.ldw;
        wx[c] = f32x4{w[0], w[1], w[2], 0.0f};
    }
    for (int c = tid; c < C2; c += NW * TK_WAVE)
        norm2[c] = constants_of(p.norm[1], c);
    for (int c = tid; c < channels; c += NW * TK_WAVE)
        norm3[c] = constants_of(p.norm[2], cbase + c);

    for (int tile = blockIdx.x; tile < a.total; tile += gridDim.x) {
        const int b = tile / a.tiles, base = (tile - b * a.tiles) * TP;
        const int pos = lane % TP;
        const int at = base + pos < P ? base + pos : P - 1;  // (results of the surplus are dropped)
        const int64_t j64 = p.index[(int64_t)b * P + at];
        const bool hit = j64 >= 0 && j64 < p.N;
        const int j = hit ? (int)j64 : 0, m = at / p.S;
        float r[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float x = p.xyz[((int64_t)b * 3 + d) * p.N + j];
            r[d] = (hit ? x : 0.0f) - p.centre[((int64_t)b * 3 + d) * p.M + m];
        }
        const float *row = p.u ? p.u + ((int64_t)b * p.N + j) * C1 : nullptr;
        const float *w2 = p.w2 + (int64_t)col * C1 + 4 * half, *w3 = p.w3 + (int64_t)(cbase + col) * C2 + 4 * half;
        const int blocks2 = C2 / 32, blocks3 = channels / 32;
        // (a wave requests the weights that it begins with before what they are multiplied with is there)
        Weights<D> now;
        if (wave < blocks2)
            now.load(w2 + (int64_t)wave * 32 * C1);
        if (tile == (int)blockIdx.x)
            __syncthreads();  // the constants
        for (int c = (wave * (TK_WAVE / TP) + lane / TP) * 8; c < C1; c += NW * (TK_WAVE / TP) * 8)
#pragma unroll
            for (int h = 0; h < 8; h += 4) {
                f32x4 v{0.0f, 0.0f, 0.0f, 0.0f};
                if (row && hit)
                    v = *reinterpret_cast<const f32x4 *>(row + c + h);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 w = wx[c + h + i];
                    v[i] = __builtin_fmaf(w.x, r[0], __builtin_fmaf(w.y, r[1], __builtin_fmaf(w.z, r[2], v[i])));
                    v[i] = relu(normalised(v[i], norm1[c + h + i]));
                }
                act1[(c + h) / 4 * ROW + pos] = v;
            }
        __syncthreads();

        for (int block = wave; block < blocks2; block += NW) {
            const float *w = w2 + (int64_t)block * 32 * C1;
            if (block != wave)
                now.load(w);
            const int channel = block * 32 + 4 * half;
            tk_f32x16 sums[PT];
            product<PT, D, ROW, true>(act1 + half * ROW + col, now, w, C1, sums);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4 v[PT];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 k = norm2[channel + 8 * q + i];
#pragma unroll
                    for (int t = 0; t < PT; ++t)
                        v[t][i] = relu(normalised(sums[t][4 * q + i], k));
                }
#pragma unroll
                for (int t = 0; t < PT; ++t)
                    act2[(channel / 4 + 2 * q) * ROW + 32 * t + col] = v[t];
            }
        }
        if (wave < blocks3)
            now.load(w3 + (int64_t)wave * 32 * C2);
        __syncthreads();

        for (int block = wave; block < blocks3; block += NW) {
            const float *w = w3 + (int64_t)block * 32 * C2;
            if (block != wave)
                now.load(w);
            const int c = block * 32 + col;
            tk_f32x16 sums[PT];
            product<PT, D, ROW, false>(act2 + half * ROW + col, now, w, C2, sums);
            const f32x4 k = norm3[c];
            float best[PT];
#pragma unroll
            for (int t = 0; t < PT; ++t) {
                best[t] = 0.0f;  // (of a ReLU)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    best[t] = __builtin_elementwise_maximum(best[t], normalised(sums[t][i], k));
                const float2 halves = tk_both_halves(best[t]);
                best[t] = __builtin_elementwise_maximum(halves.x, halves.y);
            }
            float *out = p.out + ((int64_t)b * C3 + cbase + c) * p.M;
            const int group = base / p.S;
            if (PT == 1 || p.S == TP) {
                if (half == 0)
                    out[group] = PT == 1 ? best[0] : __builtin_elementwise_maximum(best[0], best[PT - 1]);
            } else if (group + half < p.M) {
                out[group + half] = half ? best[PT - 1] : best[0];
            }
        }
    }
}

// LDS of a workgroup: both activations and the constants.
int lds_bytes(int C1, int C2, int part, int tile)
{
    return ((C1 + C2) / 4 * (tile + 1) + 2 * C1 + C2 + part) * 16;
}

constexpr int kMostLds = 155 << 10;

bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int NW, int TP> int launch(const GroupedArgs &a, int parts, hipStream_t stream)
{
    const int bytes = lds_bytes(a.p.C[0], a.p.C[1], a.part, TP);
    const int rc = tk_allow_dynamic_lds<mlp_grouped_pool_kernel<NW, TP>>(kMostLds);
    if (rc != TK3D_OK)
        return rc;
    // as many workgroups as stay on the chip at once
    const int of_lds = (160 << 10) / bytes, of_waves = 16 / NW, cu = of_lds < of_waves ? of_lds : of_waves;
    const int most = cu * tk_cu_count() / parts;
    const int grid = a.total < most ? a.total : most;
    mlp_grouped_pool_kernel<NW, TP><<<dim3(grid, parts), NW * TK_WAVE, bytes, stream>>>(a);
    return tk_launch_status();
}

// Tiles of 64 positions, which read the weights once for two products, or of 32 where those would not fill the chip
// (64 and 32, us: 8 x 32 groups of 32, 256-256-512 channels 50, 43; 1 x 128, 128-128-256 21, 16; from one tile of
// 64 per CU on 64 gains up to a third).
int64_t tiles_of(const tk3d_mlp_grouped_pool &p, int tile)
{
    return (int64_t)p.B * (((int64_t)p.M * p.S + tile - 1) / tile);
}
int pick_tile(const tk3d_mlp_grouped_pool &p) { return p.S == 32 && tiles_of(p, 64) < tk_cu_count() ? 32 : 64; }
// Eight waves share a tile if the second layer has a block of channels for every other one at least (four and
// eight, us: 32 x 777 groups of 32, 64-96-128 channels 331, 359; 32 x 128, 128-128-256 146, 143; 8 x 32,
// 256-256-512 51, 43).
int waves_of(const tk3d_mlp_grouped_pool &p) { return p.C[1] < 128 ? 4 : 8; }
// Fewer tiles than CUs: the third layer's channels over several workgroups, each of which works the first two
// layers out again (1 x 128 groups of 64, 128-128-256 channels: 24 us in one part, 21 in two, 28 in four).
int part_of(const tk3d_mlp_grouped_pool &p, int64_t tiles)
{
    const int blocks = p.C[2] / 32;
    int64_t parts = tk_cu_count() / tiles;
    parts = parts < 1 ? 1 : parts > blocks ? blocks : parts;
    return (int)((blocks + parts - 1) / parts) * 32;
}

// Whether one launch is the better choice (us, three launches and this one, 64 features in front of the first layer).
bool pays(const tk3d_mlp_grouped_pool &p)
{
    const int tile = pick_tile(p), waves = waves_of(p), cus = tk_cu_count();
    const int64_t tiles = tiles_of(p, tile);
    const int C1 = p.C[0], C2 = p.C[1], C3 = p.C[2];
    if (tiles < cus) {
        // A tile is a chain of products on one CU, which three launches spread over the chip: here the channels that a
        // wave multiplies one behind the other. A short one (two tiles of 32 at once take half as long again as one) is
        // hidden by the host's time for two launches more: a pass among others, and one that is waited for, 32 groups
        // of 64, 96-96-96 (192) 22.5, 17.4 and 35.8, 36.6; 128-128-256 (256) 22.3, 20.1 and 37.0, 38.9; with four waves
        // 192-64-64 (256) 22.7, 21.7 and 36.3, 40.8, 256-32-64 (288) 22.3, 23.9 and 36.9, 43.0; 32 of 32, 128-256-512
        // (384) 22.6, 20.5 and 37.6, 40.2; GPU time, 256-256-512 (512) 23.5, 27.7. A longer one pays with the tiles
        // that the three have to spread. GPU time, 128 groups of 64: 256-256-512 (512) 69.5, 47.3, 32-480-64 (544)
        // 35.9, 33.0; with four waves 192-64-64 (256) 23, 23, 224-32-64 (256) 21, 23, 448-64-64 (512) 33, 38; 64 groups
        // of 64, 256-256-512 (512) 37.7, 39.9.
        const auto turns = [&](int channels) { return (channels / 32 + waves - 1) / waves; };
        const int64_t chain = C1 * turns(C2) + C2 * turns(part_of(p, tiles)), all = chain * (tile / 32);
        return chain * (tile == 64 ? 3 : 2) <= (waves == 4 ? 704 : 768) ||
               (waves == 4 ? all < 4 * tiles : all <= 9 * tiles);
    }
    // Layers for which a CU holds one workgroup need work for all of its waves. A second layer of one or two blocks of
    // channels leaves most of four waves idle through the longest product: 32 x 128 groups of 64, 256-32-64 191, 289,
    // 480-32-64 367, 502, 256-64-128 267, 319 (with up to four tiles a CU two blocks gain: 16 x 32 of 32 40, 29);
    // 224-32-64, two workgroups to a CU, 174, 159. So does a third layer of one or two blocks behind a wide second one,
    // on more than four tiles a CU: 32 x 128 groups of 64, 96-256-32 270, 326, 32-480-64 380, 423, 64-256-64 248, 283;
    // 16 x 32 of 32, 96-256-32 43, 28. (128-192-32 304, 316 there and 687, 632 at 32 x 512 of 32; 256-256-512, whose
    // workgroups are alone too, 1056, 929.)
    if (2 * lds_bytes(C1, C2, C3, 64) > 160 << 10) {
        if (C2 <= 64)
            return C2 == 64 && tiles <= 4 * cus;
        if (C3 <= 64 && C2 >= 2 * C1)
            return tiles <= 4 * cus;
    }
    return true;
}

}  // namespace

extern "C" {

int tk3d_mlp_grouped_pool_supported(const tk3d_mlp_grouped_pool *p)
{
    for (int l = 0; l < 3; ++l)
        if (p->C[l] <= 0 || p->C[l] % 32 != 0 || p->C[l] > 4096)
            return 0;
    if (p->B <= 0 || p->N <= 0 || p->M <= 0 || (p->S != 32 && p->S != 64) || !tk_fits(1 << 29, p->M, p->S) ||
        tiles_of(*p, 32) > TK_MAX_I32 / 2 || lds_bytes(p->C[0], p->C[1], p->C[2], 64) > kMostLds ||
        !aligned(p->u) || !aligned(p->w2) || !aligned(p->w3))
        return 0;
    return pays(*p);
}

int tk3d_mlp_grouped_pool_f32(const tk3d_mlp_grouped_pool *p, void *stream_)
{
    if (!p)
        return TK3D_ERR_NULL_POINTER;
    if (!tk3d_mlp_grouped_pool_supported(p))
        return TK3D_ERR_UNSUPPORTED;
    const hipStream_t stream = (hipStream_t)stream_;
    const int tile = pick_tile(*p);
    GroupedArgs a;
    a.p = *p;
    a.tiles = (p->M * p->S + tile - 1) / tile;
    a.total = (int)tiles_of(*p, tile);
    a.part = part_of(*p, a.total);
    const int parts = (p->C[2] + a.part - 1) / a.part;
    if (waves_of(*p) == 4)
        return tile == 32 ? launch<4, 32>(a, parts, stream) : launch<4, 64>(a, parts, stream);
    return tile == 32 ? launch<8, 32>(a, parts, stream) : launch<8, 64>(a, parts, stream);
}

}  // extern "C"
