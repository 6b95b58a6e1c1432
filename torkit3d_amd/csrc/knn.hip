// K nearest neighbours for gfx950, returning the reference's MinK slot order.
//
// A lane owns one query and keeps its k best (distance, index) pairs in registers
// (KMAX slots, fully unrolled, no dynamic register indexing); key points are
// staged through LDS as (x,y,z,pad) quads that all lanes read as a broadcast.
// The result is not just "the k smallest": the reference returns them in the
// order its MinK structure leaves them (mink.cuh:61-89) - the first k keys fill
// slots 0..k-1, later a key that beats the current maximum (strict '<') replaces
// that maximum's slot, and the new maximum is the first slot (ascending, strict
// '>') above the inserted key. The insertion below follows that rule slot for
// slot, with selects instead of indexed writes.
//
// k above the largest register variant falls back to a kernel that keeps the
// structure in the output arrays in global memory, as the reference's generic
// variant does (knn_distance_kernel.cu:102-177).
#include <type_traits>

#include "tk3d_common.h"
#include "tk3d_curve.h"
#include "tk3d_debug.h"

namespace {

constexpr int KNN_BLOCK = 256;
constexpr int KNN_STAGE = 1024;

// Coordinate `a` of point `j` of an n-point cloud: [n,3] rows, or with SOA three planes
// [3,n] (the layout the reference's models keep their clouds in).
template <bool SOA, typename T>
__device__ __forceinline__ T knn_coord(const T *__restrict__ cloud, int n, int j, int a)
{
    return SOA ? cloud[(int64_t)a * n + j] : cloud[(int64_t)j * 3 + a];
}

// Inverse-squared-distance weights of the three neighbours, as FeatureInterpolator
// forms them with torch ops (torkit3d/layers/pointnet2.py:128-130):
// inv = 1 / clamp(d, min=eps); w = inv / (inv0 + inv1 + inv2).
template <typename T>
__device__ __forceinline__ void knn_three_weights(const T (&d)[3], T eps, T *__restrict__ w)
{
    T inv[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        inv[i] = (T)1 / (d[i] < eps ? eps : d[i]);  // a NaN stays a NaN, as in clamp
    const T norm = (inv[0] + inv[1]) + inv[2];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        w[i] = inv[i] / norm;
}

template <typename T, int KMAX, bool SOA, bool WEIGHTS>
__global__ __launch_bounds__(KNN_BLOCK) void knn_register_kernel(
    const T *__restrict__ query, const T *__restrict__ key, T *__restrict__ distance,
    int64_t *__restrict__ index, T *__restrict__ weight, T eps, int blocks_per_batch, int n1,
    int n2, int k)
{
    __shared__ T skey[KNN_STAGE * 4];
    const int tid = threadIdx.x;
    const int b = blockIdx.x / blocks_per_batch;
    const int qi = (blockIdx.x - b * blocks_per_batch) * KNN_BLOCK + tid;
    const bool active = qi < n1;
    const T *__restrict__ K = key + (int64_t)b * n2 * 3;
    T qx = 0, qy = 0, qz = 0;
    if (active) {
        const T *__restrict__ Q = query + (int64_t)b * n1 * 3;
        qx = knn_coord<SOA>(Q, n1, qi, 0);
        qy = knn_coord<SOA>(Q, n1, qi, 1);
        qz = knn_coord<SOA>(Q, n1, qi, 2);
    }

    T kd[KMAX];
    int ki[KMAX];
    T max_key = (T)0;
    int max_idx = 0;
    // Fill phase: keys 0..k-1 go to slots 0..k-1; the maximum is the first slot
    // holding the largest value (mink.cuh:63-72). Slots >= k stay at -inf so the
    // rescan below never selects them.
#pragma unroll
    for (int s = 0; s < KMAX; ++s) {
        kd[s] = -tk_inf<T>();
        ki[s] = 0;
        if (s < k) {  // uniform
            const T d = tk_dist2<T>(knn_coord<SOA>(K, n2, s, 0), knn_coord<SOA>(K, n2, s, 1),
                                       knn_coord<SOA>(K, n2, s, 2), qx, qy, qz);
            kd[s] = d;
            ki[s] = s;
            if (s == 0 || d > max_key) {
                max_key = d;
                max_idx = s;
            }
        }
    }

    for (int stage0 = 0; stage0 < n2; stage0 += KNN_STAGE) {
        __syncthreads();
        for (int j = tid; j < KNN_STAGE; j += KNN_BLOCK) {
            const int kj = stage0 + j;
            T x = 0, y = 0, z = 0;
            if (kj < n2) {
                x = knn_coord<SOA>(K, n2, kj, 0);
                y = knn_coord<SOA>(K, n2, kj, 1);
                z = knn_coord<SOA>(K, n2, kj, 2);
            }
            skey[j * 4 + 0] = x;
            skey[j * 4 + 1] = y;
            skey[j * 4 + 2] = z;
            skey[j * 4 + 3] = (T)0;
        }
        __syncthreads();
        const int left = n2 - stage0;
        const int cnt = left < KNN_STAGE ? left : KNN_STAGE;
        int j = (stage0 < k) ? (k - stage0 < cnt ? k - stage0 : cnt) : 0;
        for (; j < cnt; ++j) {
            const T d = tk_dist2<T>(skey[j * 4 + 0], skey[j * 4 + 1], skey[j * 4 + 2], qx, qy,
                                    qz);
            if (d < max_key) {
                const int kj = stage0 + j;
#pragma unroll
                for (int s = 0; s < KMAX; ++s) {
                    const bool here = (s == max_idx);
                    kd[s] = here ? d : kd[s];
                    ki[s] = here ? kj : ki[s];
                }
                max_key = d;
#pragma unroll
                for (int s = 0; s < KMAX; ++s) {
                    const bool up = kd[s] > max_key;
                    max_key = up ? kd[s] : max_key;
                    max_idx = up ? s : max_idx;
                }
            }
        }
    }

    if (active) {
        T *od = distance + ((int64_t)b * n1 + qi) * k;
        int64_t *oi = index + ((int64_t)b * n1 + qi) * k;
#pragma unroll
        for (int s = 0; s < KMAX; ++s) {
            if (s < k) {
                od[s] = kd[s];
                oi[s] = (int64_t)ki[s];
            }
        }
        if constexpr (WEIGHTS && KMAX >= 3) {  // k == 3
            const T d3[3] = {kd[0], kd[1], kd[2]};
            knn_three_weights<T>(d3, eps, weight + ((int64_t)b * n1 + qi) * 3);
        }
    }
}

// fp32 variant with batched insertion. Inserting into the k-slot structure costs a
// few dozen instructions and, done at the moment a candidate appears, is paid by the
// whole wave for every candidate of every lane. Here a lane first sweeps a chunk of
// 32 keys and only records which of them beat its current maximum (the sign of the
// integer difference of the bit patterns - non-negative floats order as integers -
// shifted into a mask: two instructions per key on top of the distance). The wave
// then inserts in rounds: every lane with a recorded candidate takes its next one
// (ascending key order), recomputes the distance, tests it against its maximum as
// it stands now (strict '<', as MinK does) and inserts. Rounds per chunk = the
// largest number of candidates any lane has, instead of the number of distinct
// candidate keys across all lanes. The sequence of insertions seen by one lane is
// exactly MinK's, so the slot order is unchanged.

// `skey` is KNN_STAGE * 4 floats of LDS, 16-byte aligned; the whole workgroup calls this
// with query `qi` of batch `b` per lane (qi >= n1: the lane only helps staging).
template <int KMAX, bool SOA, bool WEIGHTS>
__device__ __forceinline__ void knn_batched_body(
    const float *__restrict__ query, const float *__restrict__ key,
    float *__restrict__ distance, int64_t *__restrict__ index, float *__restrict__ weight,
    float eps, int b, int qi, int n1, int n2, int k, float *skey)
{
    constexpr int CHUNK = 32;
    static_assert(KNN_STAGE % CHUNK == 0, "a chunk must not straddle stages");
    const int tid = threadIdx.x;
    const bool active = qi < n1;
    const float *__restrict__ K = key + (int64_t)b * n2 * 3;
    float qx = 0, qy = 0, qz = 0;
    if (active) {
        const float *__restrict__ Q = query + (int64_t)b * n1 * 3;
        qx = knn_coord<SOA>(Q, n1, qi, 0);
        qy = knn_coord<SOA>(Q, n1, qi, 1);
        qz = knn_coord<SOA>(Q, n1, qi, 2);
    }

    float kd[KMAX];
    int ki[KMAX];
    float max_key = 0.0f;
    int max_idx = 0;
    bool fill_nan = false;
    // Fill phase: keys 0..k-1 go to slots 0..k-1 (mink.cuh:63-72); unused slots stay at
    // -inf so the rescan never selects them.
#pragma unroll
    for (int s = 0; s < KMAX; ++s) {
        kd[s] = -__builtin_huge_valf();
        ki[s] = 0;
        if (s < k) {  // uniform
            const float d = tk_dist2<float>(knn_coord<SOA>(K, n2, s, 0), knn_coord<SOA>(K, n2, s, 1),
                                       knn_coord<SOA>(K, n2, s, 2), qx, qy, qz);
            kd[s] = d;
            ki[s] = s;
            fill_nan |= d != d;
            if (s == 0 || d > max_key) {
                max_key = d;
                max_idx = s;
            }
        }
    }
    // The rescan below orders the slots by their bit patterns, which is the float order
    // for everything a squared distance can be except NaN. A NaN can only enter during
    // the fill (later keys must compare below the maximum); a wave that has one rescans
    // with float compares instead.
    const bool float_rescan = __builtin_amdgcn_ballot_w64(fill_nan) != 0;

    for (int stage0 = 0; stage0 < n2; stage0 += KNN_STAGE) {
        __syncthreads();
        for (int j = tid; j < KNN_STAGE; j += KNN_BLOCK) {
            const int kj = stage0 + j;
            float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (kj < n2) {
                e.x = knn_coord<SOA>(K, n2, kj, 0);
                e.y = knn_coord<SOA>(K, n2, kj, 1);
                e.z = knn_coord<SOA>(K, n2, kj, 2);
            }
            reinterpret_cast<float4 *>(skey)[j] = e;
        }
        __syncthreads();
        const int left = n2 - stage0;
        const int cnt = left < KNN_STAGE ? left : KNN_STAGE;
        for (int c0 = 0; c0 < cnt; c0 += CHUNK) {
            // ---- sweep: bit (31 - i) of `mask` <=> key c0+i is below the maximum ----
            const int maxbits = __builtin_bit_cast(int, max_key);
            const float4 *ck = reinterpret_cast<const float4 *>(skey) + c0;
            const int first = stage0 + c0;  // global index of bit 31
            unsigned mask = 0u;
            if (c0 + CHUNK <= cnt) {
                // A full chunk comes straight from global memory: the addresses are the
                // same for the whole wave, so the loads are scalar and the coordinates are
                // scalar operands of the vector arithmetic - no LDS traffic in the sweep.
#pragma unroll
                for (int i = 0; i < CHUNK; ++i) {
                    const float d = tk_dist2<float>(knn_coord<SOA>(K, n2, first + i, 0),
                                                    knn_coord<SOA>(K, n2, first + i, 1),
                                                    knn_coord<SOA>(K, n2, first + i, 2), qx, qy,
                                                    qz);
                    const unsigned diff = (unsigned)(__builtin_bit_cast(int, d) - maxbits);
                    mask = __builtin_amdgcn_alignbit(mask, diff, 31);  // (mask << 1) | sign
                }
            } else {
#pragma unroll 4
                for (int i = 0; i < CHUNK; ++i) {
                    const float4 e = ck[i];  // zero padding beyond the last key
                    const float d = tk_dist2<float>(e.x, e.y, e.z, qx, qy, qz);
                    const unsigned diff = (unsigned)(__builtin_bit_cast(int, d) - maxbits);
                    mask = __builtin_amdgcn_alignbit(mask, diff, 31);
                }
            }
            // Keys that do not exist, or that the fill phase took, are no candidates.
            int lo = k - first;                          // keys below k filled the slots
            lo = lo < 0 ? 0 : (lo > CHUNK ? CHUNK : lo);
            int hi = cnt - c0;                           // keys at or beyond hi are padding
            hi = hi > CHUNK ? CHUNK : hi;
            unsigned valid = (lo >= CHUNK) ? 0u : (0xffffffffu >> lo);
            valid &= (hi >= CHUNK) ? 0xffffffffu : ~(0xffffffffu >> hi);
            mask &= valid;

            // ---- insertion rounds; the next candidate's key is fetched from LDS while the
            // current one is inserted ----
            bool has = mask != 0u;
            int i = has ? __builtin_clz(mask) : 0;
            float4 e = ck[i];
            while (__builtin_amdgcn_ballot_w64(has)) {  // wave-uniform
                mask &= ~(0x80000000u >> i);  // no-op for a lane without a candidate
                const bool has_next = mask != 0u;
                const int i_next = has_next ? __builtin_clz(mask) : 0;
                const float4 e_next = ck[i_next];
                const float d = tk_dist2<float>(e.x, e.y, e.z, qx, qy, qz);
                if (has && d < max_key) {
                    const int kj = first + i;
#pragma unroll
                    for (int s = 0; s < KMAX; ++s) {
                        const bool here = (s == max_idx);
                        kd[s] = here ? d : kd[s];
                        ki[s] = here ? kj : ki[s];
                    }
                    if (float_rescan) {
                        max_key = d;
#pragma unroll
                        for (int s = 0; s < KMAX; ++s) {
                            const bool up = kd[s] > max_key;
                            max_key = up ? kd[s] : max_key;
                            max_idx = up ? s : max_idx;
                        }
                    } else {
                        // New maximum = largest bit pattern. MinK starts its rescan from the
                        // inserted key, so the maximum stays in the inserted slot when nothing
                        // is strictly above it; otherwise it is the first slot that holds the
                        // largest pattern: (top - 1 - bits) is negative exactly there, and
                        // the sign bits shifted together put slot 0 in the highest position.
                        // Both steps are written as short independent chains: with few waves
                        // per SIMD the round is bound by its dependent latency.
                        int t[KMAX];
#pragma unroll
                        for (int s = 0; s < KMAX; ++s)
                            t[s] = __builtin_bit_cast(int, kd[s]);
#pragma unroll
                        for (int n = KMAX; n > 1; n = (n + 2) / 3) {
#pragma unroll
                            for (int j = 0; 3 * j < n; ++j) {
                                int v = t[3 * j];
                                if (3 * j + 1 < n)
                                    v = t[3 * j + 1] > v ? t[3 * j + 1] : v;
                                if (3 * j + 2 < n)
                                    v = t[3 * j + 2] > v ? t[3 * j + 2] : v;
                                t[j] = v;
                            }
                        }
                        const int top = t[0];
                        const unsigned below = (unsigned)top - 1u;
                        constexpr int GS = KMAX <= 16 ? 4 : 8;  // slots per independent chain
                        unsigned eq[(KMAX + 31) / 32] = {};
#pragma unroll
                        for (int g0 = 0; g0 < KMAX; g0 += GS) {
                            unsigned part = 0u;
#pragma unroll
                            for (int s = g0; s < g0 + GS; ++s)
                                part = __builtin_amdgcn_alignbit(
                                    part, below - __builtin_bit_cast(unsigned, kd[s]), 31);
                            eq[g0 / 32] = (eq[g0 / 32] << GS) | part;
                        }
                        max_key = __builtin_bit_cast(float, top);
                        int first_top;
                        if constexpr (KMAX <= 32)
                            first_top = __builtin_clz(eq[0]) - (32 - KMAX);
                        else
                            first_top = eq[0] ? __builtin_clz(eq[0]) : 32 + __builtin_clz(eq[1]);
                        max_idx = top != __builtin_bit_cast(int, d) ? first_top : max_idx;
                    }
                }
                has = has_next;
                i = i_next;
                e = e_next;
            }
        }
    }

    if (active) {
        float *od = distance + ((int64_t)b * n1 + qi) * k;
        int64_t *oi = index + ((int64_t)b * n1 + qi) * k;
#pragma unroll
        for (int s = 0; s < KMAX; ++s) {
            if (s < k) {
                od[s] = kd[s];
                oi[s] = (int64_t)ki[s];
            }
        }
        if constexpr (WEIGHTS && KMAX >= 3) {  // k == 3
            const float d3[3] = {kd[0], kd[1], kd[2]};
            knn_three_weights<float>(d3, eps, weight + ((int64_t)b * n1 + qi) * 3);
        }
    }
}

template <int KMAX, bool SOA, bool WEIGHTS>
__global__ __launch_bounds__(KNN_BLOCK) void knn_batched_kernel_f32(
    const float *__restrict__ query, const float *__restrict__ key,
    float *__restrict__ distance, int64_t *__restrict__ index, float *__restrict__ weight,
    float eps, int blocks_per_batch, int n1, int n2, int k)
{
    __shared__ __align__(16) float skey[KNN_STAGE * 4];
    const int b = blockIdx.x / blocks_per_batch;
    const int qi = (blockIdx.x - b * blocks_per_batch) * KNN_BLOCK + threadIdx.x;
    knn_batched_body<KMAX, SOA, WEIGHTS>(query, key, distance, index, weight, eps, b, qi, n1, n2,
                                         k, skey);
}

// A slot of the sorted list below: the bit pattern of the distance above (flag, KMAX - 1 - slot, key
// index). As a double it orders by distance and, among equal distances, by the low word: no pattern of
// a float is one of a NaN or an infinity up there, zero is a (kept) subnormal, the negative patterns
// of the placeholders are below all others.
template <int KMAX> struct KnnSlot {
    static constexpr int SLOT_BITS = KMAX == 64 ? 6 : KMAX == 32 ? 5 : KMAX == 16 ? 4 : KMAX == 8 ? 3 : 2;
    static constexpr int KEY_BITS = 31 - SLOT_BITS;
    static constexpr unsigned FLAG = 0x80000000u;
    static constexpr unsigned SLOT = (unsigned)(KMAX - 1) << KEY_BITS;  // mask of the slot's bits
    static constexpr unsigned KEY = (1u << KEY_BITS) - 1u;
    static_assert((1 << SLOT_BITS) == KMAX, "4 to 64 slots");
    static __device__ __forceinline__ double pack(int distance, unsigned low)
    {
        return __builtin_bit_cast(double, ((unsigned long long)(unsigned)distance << 32) | low);
    }
    static __device__ __forceinline__ int distance(double v)
    {
        return (int)(__builtin_bit_cast(unsigned long long, v) >> 32);
    }
    static __device__ __forceinline__ unsigned low(double v)
    {
        return (unsigned)__builtin_bit_cast(unsigned long long, v);
    }
    static __device__ __forceinline__ int slot(double v)
    {
        return KMAX - 1 - (int)((low(v) & SLOT) >> KEY_BITS);
    }
};

// (written out as tk_min_f64 is)
__device__ __forceinline__ double knn_min_f64_uniform(double a, double b)  // b wave-uniform
{
    double o;
    asm("v_min_f64 %0, %1, %2" : "=v"(o) : "v"(a), "s"(b));
    return o;
}
__device__ __forceinline__ double knn_max_f64(double a, double b)
{
    double o;
    asm("v_max_f64 %0, %1, %2" : "=v"(o) : "v"(a), "v"(b));
    return o;
}

// fp32, k <= 32, launches with many queries: pre-filtered sweep with deferred insertions.
//
// Two costs dominate the batched kernel above: its sweep spends 8 vector instructions per
// pair (six for the canonical distance), and its insertion rounds run after every chunk
// for as long as the slowest lane of the wave has candidates, most lanes idling.
//
// Sweep. As in the chamfer kernel, most pairs only need to be ruled out, which the score
//     s(q,k) = |k'|^2 - 2 q'.k'      (k' = k - c, q' = q - c, c the centre of the key
//                                      cloud's bounding box)
// does: d2(q,k) = s + |q'|^2 up to rounding. A key can only be inserted if its canonical
// distance is below the query's current maximum M, so the sweep takes the sign of t = s - thr,
// thr = (M - |q'|^2) + slack: candidates are the keys with t < 0. The scores come from the matrix
// cores: one v_mfma_f32_32x32x16_f16 gives t for 32 keys x 32 queries as a 16-term dot product of
// fp16 pieces, and a lane only has to collect the 16 sign bits it is handed (1.1 vector
// instructions per pair). Coordinates are centred and multiplied by a power of two that brings
// half the diagonal of the keys' bounding box, which no centred key norm exceeds, into [2, 4) (exact; outside
// 2^-40 .. 2^40 the workgroup takes the exact sweep; a key lies on the box's longest side, 2 / sqrt(3) or more from
// the centre), then split into two fp16 pieces each, x = xh + xl + e with |e| <= 2^-23 |x| +
// 2^-25, |k'|^2 into two and -thr into two:
//     key   : xh xh xl  yh yh yl  1  1  | zh zh zl  n0 n1 0  1  1
//     query : Xh Xl Xh  Yh Yl Yh  T0 T1 | Zh Zl Zh  1  1  0  T0 T1        (X = -2 q'x)
// In the 32 x 32 result lane l holds rows (keys) 16 h .. 16 h + 15, h = l / 32, of column
// (query) l % 32; lane l puts the key of that row into the tile, so the sign bits of a
// lane are 16 consecutive bits of the chunk mask. The wave's 64 queries are two blocks of 32,
// block h the queries of the lanes of half h; a lane computes its thr and writes -thr into the T
// terms of its own half only (the other half holds zeros there), so no thr crosses lanes; the
// halves of a mask meet through one exchange of registers between lanes l and l ^ 32. With
// u = 2^-24, rho = |k'| + |q'|, R = (max|k'| + |q'|)^2, in the rescaled units:
//     canonical d2 against the exact distance of the centred points   7.02 u rho^2
//         (three rounded differences, a product and two fmas of non-negative terms,
//          plus the rounding of k' and q' themselves)
//     |k'|^2 as staged, thr itself                         3 u |k'|^2 + 3 u (M + R)
//     pieces dropped from 2 q'.k', subnormal pieces                       5 u R
//     |k'|^2 and thr in two pieces                           4 u R + 4 u (M + R)
//     the matrix core's 16 additions: 32 u times the sum of the products' magnitudes
//         as the matrix core sees them (a subnormal fp16 factor counts as 2^-14; see
//         the chamfer kernel and tests/test_gpu_mfma_bound.py), which is below
//         1.02 (M + R) here because the scale makes max|k'| > 1      33 u (M + R)
// below 59 u R + 40 u M; the kernel uses slack = 64 u R + 48 u M (+1e-37 against underflow), R from
// the bound of |k'| and |q'| inflated by 1e-6 for their own rounding. Every key with canonical d2 < M
// therefore has t < 0: the sign bits are a superset of MinK's insertions. Queries further than 200
// from the centre (rescaled; thr would leave fp16's range) take every key as a candidate, key clouds
// that are non-finite or huge the exact batched sweep.
//
// Boxes. In launches with keys enough (knn_filter_launch) the workgroup's 512 queries are sorted along a Hilbert
// curve, so that a wave has neighbours: its 64 queries' box is small, and a key whose distance to that box - by the
// operations of the canonical distance on the per-axis gaps, each of which is monotone, hence a bound for every query
// in the box - is not below the largest of the wave's maxima is a candidate of none of them. A lane tests a key, and
// what passes goes into the wave's list in LDS, in key order; the sweep takes its chunks of 32 from there. Of 2048
// keys 780 pass for waves of 512 sorted queries at k = 3 and 1050 at k = 16 (sorted along a Morton curve 980 and
// 1190; 8192 queries sorted together 300 and 470, but they take a kernel and a workspace of their own). Of fewer keys
// too many pass, and of 256 sorted queries a wave's box is too large. Where every key is swept its own number is its
// place in the list, which is then not written down.
//
// Keys in an order - scan lines, voxels - come near one wave of sorted queries at a time, and the others wait for it
// at the barrier of each stage, with no second workgroup on the CU to use it. A workgroup that may be alone on its CU
// therefore compares the box of the first stage's keys with that of all: in random order 512 of 2^16 normally
// distributed keys reach over about 0.7 of the cloud, in the order of a coordinate or a space-filling curve 512 of
// 1024 keys over half of an axis and of more over less. Under 0.6, it sweeps every key for its queries as they come
// (and half of them, where CUs would be left without a workgroup: the other half has one of its own, which otherwise
// ends there). us, 8 x 4096 queries, keys by x and by the voxels of a 16^3 grid along a Morton curve, without this
// test, with it: 4096 keys k = 3 131, 101 and 332, 253, k = 8 177, 129 and 483, 336; 8192 keys k = 16 396, 288 and
// 1206, 904; it takes 0 to 3 % of the time on keys in random order. Two workgroups to a CU fill each other's waits,
// and are left with the boxes: 32 x 8192 on 4096 in voxels k = 3 422, every key 471, by x 194 and 194.
//
// The first keys behind the fill are below the maximum of half of the queries or more: up to 3 k (2 k with 32 slots) they
// are put to all of them, without a sweep and a queue (a third less work than the steps they save: 142 -> 109 of
// them at k = 16).
//
// Insertions. A candidate is re-evaluated with the canonical arithmetic and inserted
// under MinK's strict test against the maximum as it stands then, in ascending key
// order per query, so the slots go through exactly MinK's states. But insertion does not
// follow every chunk: a lane keeps up to CAP non-empty chunk masks in a small
// register queue and the wave runs a service step (every lane with a pending candidate
// takes its first one) only while some lane holds T candidates or a full queue; the
// rest waits for company. Deferring only makes M - and with it thr - a little stale,
// i.e. admits more candidates, each rejected by the strict test when it is served.
//
// Slots. They are kept in descending order, each a double made of the distance's bit pattern above
// (flag, KMAX - 1 - slot, key index): v_min_f64 and v_max_f64 run at the rate of 32-bit
// instructions, compare both words at once and need no selects, so an insertion (the head leaves, x sinks
// to its place: position p becomes the larger of its lower neighbour and the smaller of itself and
// x) is 2 KMAX - 1 instructions, slot numbers, key indices and ties included. MinK's order among equal
// distances (mink.cuh:74-87: the rescan starts from the inserted key and moves on only to a strictly
// larger one, so the maximum is the inserted slot if nothing is strictly above it, else the lowest slot
// holding the largest distance) is the order of the low words - equal distances in ascending slot
// order - except that a key with nothing strictly above it goes to the head: it gets the flag, which
// leaves with it at the next insertion. 64 instructions a step at k = 16 where a list of distances with
// the slot numbers as nibbles of a 64-bit word and the key indices in LDS took 86 (a median per
// position, a binary search, the nibbles' rotation), and 40 at k = 3 where slots in registers in their
// own order took 112 (selects, a maximum, a scan for its first slot).
//
// Bound by vector issue, of which the steps are half to two thirds: a lane is a query whose candidates are served in
// key order, so 59 % of the lanes are busy in a step at k = 16, a third at k = 3. 512 lanes share the staged keys and
// the sort (up to 126 registers and 66 KB of LDS, 50 without boxes: four waves per SIMD); 32 slots run in 256, of
// which a CU holds three workgroups (with boxes of 256 queries they took up to 1.13 times as long: 80 x 250 on 16384
// in clusters k = 20 328, 291 without). us, every key swept and none put
// to all queries, and now: 32 x 8192 queries on 2048 keys k = 3 63.5, 49.5, k = 8 83, 69, k = 16 122, 110, k = 32
// 262, 246; 8 x 4096 on 16384 k = 3 214, 139, k = 16 251, 198; 8 x 4096 on 256 k = 3 15.3, 12.9, k = 16 28.2, 25.4;
// 200 x 120 on 4096 k = 8 66, 60.
enum { KNN_EVERY_KEY, KNN_BOXES, KNN_BOXES_UNLESS_ORDERED };  // (what is passed over)

constexpr int knn_max4(int a, int b, int c, int d)
{
    const int ab = a > b ? a : b, cd = c > d ? c : d;
    return ab > cd ? ab : cd;
}

// The places of all cells of an 8^3 grid along a Hilbert curve.
struct KnnCurve {
    unsigned short place[512];
};
constexpr KnnCurve knn_make_curve()
{
    KnnCurve t{};
    for (unsigned i = 0; i < 512u; ++i)  // (eight neighbours along the curve of 16^3 are a cell of 8^3)
        t.place[i] = (unsigned short)(tk_hilbert(2u * (i >> 6), 2u * ((i >> 3) & 7u), 2u * (i & 7u)) >> 3);
    return t;
}
__device__ constexpr KnnCurve knn_curve alignas(16) = knn_make_curve();

template <int KMAX, int LANES> struct KnnFilter {
    static constexpr int BLOCK = LANES;
    static constexpr int NW = BLOCK / TK_WAVE;
    static constexpr int STAGE = KMAX > 16 ? 256 : 512;
    static constexpr int PER = STAGE / BLOCK;
    static constexpr int CHUNK = 32;
    static constexpr int RING = 2 * STAGE;  // a wave's list: it goes back to the first key of the stage before
    static constexpr int CELLS = 512;
    // Two stage buffers of key terms, [key][half] x 16 bytes, then two of raw keys (x, y, z, number) for the
    // boxes' test and the service steps; before them the sort's counters, behind them the results.
    static constexpr int SCORE_FLOATS = 2 * STAGE * 8;
    static constexpr int STAGING_FLOATS = SCORE_FLOATS + 2 * STAGE * 4;
    static constexpr int SORT_FLOATS = CELLS + 4 + CELLS / 2 + 4 * BLOCK;
    // rows of results that leave together (36 KB of LDS with 8 slots, 40 at most)
    static constexpr int ROW = KMAX + 1;
    static constexpr int ROWS_FIT = KMAX == 4 ? 1024 : 4096 / KMAX;
    static constexpr int ROWS = ROWS_FIT < BLOCK ? ROWS_FIT : BLOCK;
    static constexpr int LDS_FLOATS = knn_max4(STAGING_FLOATS, ROWS * ROW * 2, SORT_FLOATS, KNN_STAGE * 4);
    static constexpr int RED = 19;  // words a wave leaves to the others
    static_assert(STAGE % BLOCK == 0, "stage shape");
};

// -lowest and highest of each axis
__device__ __forceinline__ void knn_reach_out(float (&e)[6], const float (&v)[3])
{
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        e[a] = __builtin_fmaxf(e[a], -v[a]);
        e[3 + a] = __builtin_fmaxf(e[3 + a], v[a]);
    }
}

// The lane's keys of stage `st`. (Past the end: in no box's reach, and of no chunk's.)
template <bool SOA, int PER, int BLOCK>
__device__ __forceinline__ void knn_filter_fetch(float4 (&pre)[PER], const float *__restrict__ K, int n2, int st)
{
    const float INF = __builtin_huge_valf();
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int kj = (st * PER + r) * BLOCK + (int)threadIdx.x;
        pre[r] = make_float4(INF, INF, INF, __builtin_bit_cast(float, kj));
        if (kj < n2)
            pre[r] = make_float4(knn_coord<SOA>(K, n2, kj, 0), knn_coord<SOA>(K, n2, kj, 1),
                                 knn_coord<SOA>(K, n2, kj, 2), __builtin_bit_cast(float, kj));
    }
}

// What the kernel has found out before it comes to its queries.
template <int PER> struct KnnFrame {
    float centre[3], scale, kmax;   // of the keys; kmax bounds their rescaled norms
    float origin[3], cells[3];      // of the grid that sorts the queries, with boxes
    float own[3];                   // the lane's query before that
    float4 pre[PER];                // the lane's keys of the first stage
};

// The queries base .. base + span - 1 of cloud b, a lane each; BOXES: sorted, keys outside a wave's box passed over.
template <int KMAX, bool SOA, bool WEIGHTS, int LANES, bool BOXES>
__device__ __forceinline__ void knn_filter_queries(
    const float *__restrict__ Q, const float *__restrict__ K, float *__restrict__ distance,
    int64_t *__restrict__ index, float *__restrict__ weight, float eps, int b, int base, int span, int n1, int n2, int k,
    KnnFrame<KnnFilter<KMAX, LANES>::PER> &frame, float *skey, unsigned short *rings,
    float (*sred)[KnnFilter<KMAX, LANES>::RED])
{
    using F = KnnFilter<KMAX, LANES>;
    using Slot = KnnSlot<KMAX>;
    constexpr int BLOCK = F::BLOCK, NW = F::NW, STAGE = F::STAGE, PER = F::PER, CHUNK = F::CHUNK, RING = F::RING;
    constexpr int CELLS = F::CELLS, ROW = F::ROW, ROWS = F::ROWS;
    constexpr int TEST = 2;  // keys a lane tests against the box at once
    constexpr int CAP = 4;
    constexpr int T = 6;
    static_assert(!WEIGHTS || KMAX == 4, "weights of three neighbours");
    static_assert(!BOXES || (3 * KMAX <= TK_WAVE && STAGE % (TEST * TK_WAVE) == 0 && CELLS == BLOCK), "boxes' shape");
    float4 *const sraw = reinterpret_cast<float4 *>(skey + F::SCORE_FLOATS);
    uint4 *const sterm = reinterpret_cast<uint4 *>(skey);
    const int tid = threadIdx.x;
    const int lane = tid & (TK_WAVE - 1);
    const int half = (tid >> 5) & 1;
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE);
    const float INF = __builtin_huge_valf();
    const float c0 = frame.centre[0], c1 = frame.centre[1], c2 = frame.centre[2];
    const float scale = frame.scale, kmax = frame.kmax;
    const float scale2 = scale * scale;  // <= 2^82
    const int nstages = (n2 + STAGE - 1) / STAGE;

    // ---- the workgroup's queries in the order of their cells along a Hilbert curve, those that do not exist last
    // (a counting sort; the order within a cell is whatever the atomics give, which no result depends on) ----
    int mine = tid;
    float qx = frame.own[0], qy = frame.own[1], qz = frame.own[2];
    if constexpr (BOXES) {
        unsigned *const cnt = reinterpret_cast<unsigned *>(skey);
        const unsigned short *const curve = reinterpret_cast<const unsigned short *>(cnt + CELLS + 4);
        float4 *const order = reinterpret_cast<float4 *>(cnt + CELLS + 4 + CELLS / 2);
        unsigned cell = CELLS;
        if (base + tid < n1) {
            unsigned at = 0u;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float f = (frame.own[a] - frame.origin[a]) * frame.cells[a];
                // (a NaN or an out-of-range value lands in cell 0 or 7)
                at = 8u * at + (unsigned)(int)__builtin_fminf(__builtin_fmaxf(f, 0.0f), 7.0f);
            }
            cell = curve[at];
        }
        const unsigned turn = atomicAdd(&cnt[cell], 1u);
        __syncthreads();
        const unsigned sum = cnt[tid];  // (a cell to a lane)
        unsigned incl = sum;
#pragma unroll
        for (int o = 1; o < TK_WAVE; o <<= 1) {
            const unsigned up = (unsigned)__shfl_up((int)incl, o);
            incl += lane >= o ? up : 0u;
        }
        if (lane == TK_WAVE - 1)
            sred[wave][18] = __builtin_bit_cast(float, incl);
        __syncthreads();
        unsigned start = incl;
#pragma unroll
        for (int w = 0; w < NW; ++w)
            start += w < wave ? __builtin_bit_cast(unsigned, sred[w][18]) : 0u;
        cnt[tid] = start - sum;
        if (tid == BLOCK - 1)
            cnt[CELLS] = start;
        __syncthreads();
        order[cnt[cell] + turn] = make_float4(qx, qy, qz, __builtin_bit_cast(float, tid));
        __syncthreads();
        const float4 q = order[tid];
        qx = q.x;
        qy = q.y;
        qz = q.z;
        mine = __builtin_bit_cast(int, q.w);
    }

    // ---- the lane's query ----
    const int qi = base + mine;
    const bool active = mine < span && qi < n1;
    if (!BOXES && active) {
        qx = knn_coord<SOA>(Q, n1, qi, 0);
        qy = knn_coord<SOA>(Q, n1, qi, 1);
        qz = knn_coord<SOA>(Q, n1, qi, 2);
    }
    // the box of the wave's queries
    float box[6] = {-INF, -INF, -INF, -INF, -INF, -INF};
    if constexpr (BOXES) {
        if (active) {
            const float v[3] = {qx, qy, qz};
            knn_reach_out(box, v);
        }
        tk_wave_max_six<64>(box);
#pragma unroll
        for (int a = 0; a < 6; ++a)
            box[a] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, box[a]), TK_WAVE - 1));
    }
    float qn, slack_r;
    bool usable;
    // The query side of the 16 terms for the wave's two blocks of 32 queries, block h being the
    // queries of the lanes of half h. This lane supplies terms 8 half .. 8 half + 7 of column
    // lane % 32 in either block, from its own coordinates or, for the other half's block, its
    // partner's. The T terms (.w) are written whenever the maximum has changed.
    uint4 qterm[2];
    {
        const float px = (qx - c0) * scale, py = (qy - c1) * scale, pz = (qz - c2) * scale;
        qn = __builtin_fmaf(pz, pz, __builtin_fmaf(py, py, px * px));
        const float qnorm = __builtin_sqrtf(qn) * 1.000001f;
        const float r = kmax + qnorm;
        slack_r = r * r * 3.8146973e-06f + 1e-37f * scale2;  // 64 u R
        usable = qnorm <= 200.0f;                            // false for NaN
        const float ax = usable ? -2.0f * px : 0.0f, ay = usable ? -2.0f * py : 0.0f,
                    az = usable ? -2.0f * pz : 0.0f;
        const float ox = __shfl_xor(ax, 32), oy = __shfl_xor(ay, 32), oz = __shfl_xor(az, 32);
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const bool own = half == hb;
            const float X = own ? ax : ox, Y = own ? ay : oy, Z = own ? az : oz;
            const unsigned sx = tk_f16_split2(X), sy = tk_f16_split2(Y), sz = tk_f16_split2(Z);
            const unsigned xh = sx & 0xffffu, yh = sy & 0xffffu, zh = sz & 0xffffu;
            qterm[hb] = half == 0 ? make_uint4(sx, xh | (yh << 16), (sy >> 16) | (yh << 16), 0u)
                                  : make_uint4(sz, zh | 0x3c000000u, 0x00003c00u, 0u);
        }
    }

    // ---- the slots, in descending order of their distances. A NaN can only enter during the
    // fill (a later key must compare below the maximum) and MinK never selects such a slot as
    // maximum unless it is slot 0, in which case it never inserts again: here a NaN slot holds
    // the pattern of -inf (below every distance) and is recomputed when the results are written,
    // and a NaN in slot 0 freezes the query (maximum -inf: no key compares below it). Unused
    // slots hold the double's -inf, below all others. ----
    constexpr int NEG_INF_BITS = (int)0xff800000u;
    const double UNUSED = -__builtin_huge_val();
    double v[KMAX];
    unsigned nan_slots = 0u;
    bool frozen = false;
#pragma unroll
    for (int s = 0; s < KMAX; ++s)
        v[s] = UNUSED;
    float max_key = 0.0f;
    // Pending chunk masks, oldest first (bit 31 = first key of the chunk), and the place in the wave's list
    // of bit 31 of each, without a list the key. Named and no loops over the queue, so it stays in registers.
    static_assert(CAP == 4, "the queue is written out for four entries");
    unsigned m0 = 0u, m1 = 0u, m2 = 0u, m3 = 0u;
    int b0 = 0, b1 = 0, b2 = 0, b3 = 0;
    int qlen = 0, pending = 0;

    // The wave's list: 16 times which key of the two buffers. Where boxes pass nothing over it has every key at its own
    // number, and is not written down. (A place that nothing was listed at is read where a query has no candidate.)
    unsigned short *const ring = rings + (BOXES ? wave * (RING + CHUNK) : 0);
    unsigned char *const lds_raw = reinterpret_cast<unsigned char *>(sraw);
    unsigned char *const lds_term = reinterpret_cast<unsigned char *>(sterm);
    if constexpr (BOXES)
        for (int i = lane; i < (RING + CHUNK) / 8; i += TK_WAVE)
            reinterpret_cast<uint4 *>(ring)[i] = make_uint4(0u, 0u, 0u, 0u);
    const auto listed = [&](int i) { return BOXES ? (int)ring[i] : 16 * (i & (RING - 1)); };
    int head = 0, tail = 0;  // places of the list: swept up to, filled up to (uniform)

    // Puts a key to the lane's query.
    auto put = [&](const float4 &raw, int kj, bool has) {
        const float d = tk_dist2<float>(raw.x, raw.y, raw.z, qx, qy, qz);
        const bool ins = has && d < max_key;  // MinK's strict test (mink.cuh:74)
        const int dbits = __builtin_bit_cast(int, d);
        // The key takes the slot of the maximum, which leaves. With nothing that stays strictly
        // above it, it is the next maximum: the flag puts it in front of its equals. A key that is
        // not inserted sinks nowhere: above every pattern.
        const unsigned low = (Slot::low(v[0]) & Slot::SLOT) | (unsigned)kj;
        const unsigned flag = dbits >= Slot::distance(v[1]) ? Slot::FLAG : 0u;
        const double x = Slot::pack(ins ? dbits : 0x7fe00000, low | flag);
#pragma unroll
        for (int p = 0; p < KMAX - 1; ++p)
            v[p] = knn_max_f64(v[p + 1], tk_min_f64(v[p], x));
        v[KMAX - 1] = tk_min_f64(v[KMAX - 1], x);
        max_key = ins ? __builtin_bit_cast(float, Slot::distance(v[0])) : max_key;
    };

    // One service step: every query with a pending candidate takes its first one.
    auto service = [&]() {
        const bool has = qlen > 0;
        // (an empty queue has m0 == 0: the bit number is then meaningless, the address
        // below stays inside the buffer and nothing is inserted)
        const int bit = __builtin_clz(m0 | 1u);
        // resident: candidates are never older than the previous stage (see below)
        const float4 raw = *reinterpret_cast<const float4 *>(lds_raw + listed(b0 + bit));
        const int kj = __builtin_bit_cast(int, raw.w);
        const unsigned rest = m0 & ~(0x80000000u >> bit);
        const bool shift = has && rest == 0u;
        m0 = shift ? m1 : rest;
        b0 = shift ? b1 : b0;
        m1 = shift ? m2 : m1;
        b1 = shift ? b2 : b1;
        m2 = shift ? m3 : m2;
        b2 = shift ? b3 : b2;
        m3 = shift ? 0u : m3;
        qlen -= shift ? 1 : 0;
        pending -= has ? 1 : 0;
        put(raw, kj, has);
        // Keep the loop-carried state where it is: without this the register allocator
        // rotates some forty values through copies on every step.
        asm volatile("" : "+v"(m0), "+v"(m1), "+v"(m2), "+v"(m3));
        asm volatile("" : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3));
        asm volatile("" : "+v"(qlen), "+v"(pending), "+v"(max_key));
#pragma unroll
        for (int s = 0; s < KMAX; ++s)
            asm volatile("" : "+v"(v[s]));
    };
    auto must_serve = [&]() {
        return __builtin_amdgcn_ballot_w64(pending >= T || qlen >= CAP) != 0;
    };

    // ---- sweep: keys centred and staged in two LDS buffers, one barrier per stage ----
    auto stash = [&](int buf) {
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int j = buf * STAGE + r * BLOCK + tid;
            const float ex = frame.pre[r].x - c0, ey = frame.pre[r].y - c1, ez = frame.pre[r].z - c2;
            const float x = ex * scale, y = ey * scale, z = ez * scale;
            const float n = __builtin_fmaf(ez, ez, __builtin_fmaf(ey, ey, ex * ex)) * scale2;
            const unsigned sx = tk_f16_split2(x), sy = tk_f16_split2(y), sz = tk_f16_split2(z);
            const unsigned xh = sx & 0xffffu, yh = sy & 0xffffu, zh = sz & 0xffffu;
            const unsigned sn = tk_f16_split2(n);
            sterm[2 * j] = make_uint4(xh * 0x10001u, (sx >> 16) | (yh << 16), yh | (sy & 0xffff0000u),
                                      0x3c003c00u);
            sterm[2 * j + 1] = make_uint4(zh * 0x10001u, (sz >> 16) | (sn << 16), sn >> 16, 0x3c003c00u);
            sraw[j] = frame.pre[r];
        }
    };
    bool stale = true;    // the T terms do not belong to the maximum any more
    bool moved = true;    // nor does the wave's reach
    float reach = 0.0f;   // the largest of the queries' maxima
    // The key of a chunk in this lane's row of the tile: lane half h of the result holds rows 8 a + 4 h + c.
    const int row = (lane & 3) | ((lane >> 1) & 12) | ((lane & 4) << 2);
    // Sweeps the next `count` <= 32 keys of the list, and serves what has to be.
    auto sweep = [&](int count) {
        tk_wave_fence();  // (the list is the wave's own)
        const int first = head & (RING - 1);  // (a chunk goes on into the ring's beginning behind its end)
        const int at = listed(first + (row < count ? row : 0));
        const tk_f16x8 ka = *reinterpret_cast<const tk_f16x8 *>(lds_term + 2 * at + 16 * half);
        if (stale) {  // uniform
            const float m = max_key * scale2;  // rescaled units; slack 64 u R + 48 u M
            const float thr = (m - qn) + __builtin_fmaf(m, 2.8610229e-06f, slack_r);
            const unsigned tp = tk_f16_split2(-thr);
            qterm[0].w = half == 0 ? tp : 0u;
            qterm[1].w = half == 1 ? tp : 0u;
            stale = false;
        }
        unsigned m16[2];
        const tk_f32x16 zero = {};
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const tk_f32x16 acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                ka, __builtin_bit_cast(tk_f16x8, qterm[g]), zero, 0, 0, 0);
            unsigned m = 0u;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float t = acc[r];  // (a bit_cast applied to acc[r] itself reads element 0)
                m = __builtin_amdgcn_alignbit(m, __builtin_bit_cast(unsigned, t), 31);
            }
            m16[g] = m;
        }
        // Lane l has rows (keys) 16 half .. of column l % 32 of both blocks, the first key in
        // the highest bit. The upper lanes of block 0 change places with the lower ones of
        // block 1: then it has both halves of the rows of its own column of its own block.
        const auto both = __builtin_amdgcn_permlane32_swap(m16[0], m16[1], false, false);
        const unsigned mask = ((unsigned)both[0] << 16) | (unsigned)both[1];
        const unsigned valid = ~(unsigned)(0xffffffffull >> count);
        const unsigned m = active ? (usable ? mask : 0xffffffffu) & valid : 0u;
        const bool nz = m != 0u;
        const int to = nz ? qlen : -1;
        m0 = to == 0 ? m : m0;
        b0 = to == 0 ? first : b0;
        m1 = to == 1 ? m : m1;
        b1 = to == 1 ? first : b1;
        m2 = to == 2 ? m : m2;
        b2 = to == 2 ? first : b2;
        m3 = to == 3 ? m : m3;
        b3 = to == 3 ? first : b3;
        qlen += nz ? 1 : 0;
        pending += __builtin_popcount(m);
        head += count;
        // (two steps per trip: the loop-carried state is copied between registers once
        // per trip, some forty moves)
        while (must_serve()) {
            stale = moved = true;
            service();
            if (!must_serve())
                break;
            service();
        }
    };
    __syncthreads();
    stash(0);
    __syncthreads();
    // fill: keys 0..k-1 go to slots 0..k-1 (mink.cuh:63-72)
#pragma unroll
    for (int s = 0; s < KMAX; ++s) {
        if (s < k) {  // uniform
            const float4 raw = sraw[s];
            const float d = tk_dist2<float>(raw.x, raw.y, raw.z, qx, qy, qz);
            const bool isnan = d != d;
            nan_slots |= isnan ? (1u << s) : 0u;
            frozen |= isnan && s == 0;
            const double x = Slot::pack(isnan ? NEG_INF_BITS : __builtin_bit_cast(int, d),
                                        ((unsigned)(KMAX - 1 - s) << Slot::KEY_BITS) | (unsigned)s);
#pragma unroll
            for (int p = s; p >= 1; --p)
                v[p] = knn_max_f64(v[p], tk_min_f64(v[p - 1], x));
            v[0] = knn_max_f64(v[0], x);
        }
    }
    max_key = frozen ? -INF : __builtin_bit_cast(float, Slot::distance(v[0]));
    int before = 0;  // where the list was when this stage began
    // The first keys behind the fill are below the maximum of so many queries that they are put to all of them.
    const int taken_fit = KMAX <= 16 ? 3 * k : 2 * k;
    const int taken = taken_fit < n2 ? taken_fit : n2;
    for (int j = k; j < taken; ++j) {
        const float4 raw = sraw[j];
        put(raw, j, active);
    }
    const bool idle = __builtin_amdgcn_ballot_w64(active) == 0;  // (a wave of queries that do not exist)
    if (!BOXES)
        head = tail = taken;
    for (int st = 0; st < nstages; ++st) {
        const int stage0 = st * STAGE, buf = (st & 1) * STAGE;
        if (st + 1 < nstages)
            knn_filter_fetch<SOA, PER, BLOCK>(frame.pre, K, n2, st + 1);
        const int left = n2 - stage0;
        const int cnt = left < STAGE ? left : STAGE;
        // (without boxes a stage at a time)
#pragma unroll 1
        for (int j0 = 0; j0 < cnt; j0 += BOXES ? TEST * TK_WAVE : STAGE) {
            if constexpr (BOXES) {
                if (moved) {  // uniform
                    reach = tk_wave_extreme<true>(active ? max_key : -INF);
                    moved = false;
                }
                float4 raw[TEST];
                unsigned long long in[TEST];
#pragma unroll
                for (int u = 0; u < TEST; ++u)
                    raw[u] = sraw[buf + j0 + u * TK_WAVE + lane];
#pragma unroll
                for (int u = 0; u < TEST; ++u) {
                    // (box[a] is -lowest)
                    const float gx = __builtin_fmaxf(__builtin_fmaxf(-box[0] - raw[u].x, raw[u].x - box[3]), 0.0f);
                    const float gy = __builtin_fmaxf(__builtin_fmaxf(-box[1] - raw[u].y, raw[u].y - box[4]), 0.0f);
                    const float gz = __builtin_fmaxf(__builtin_fmaxf(-box[2] - raw[u].z, raw[u].z - box[5]), 0.0f);
                    const float bound = __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
                    in[u] = __builtin_amdgcn_ballot_w64(bound < reach);
                }
                if (st == 0 && j0 == 0)  // uniform; these have been taken
                    in[0] = taken < TK_WAVE ? in[0] & (~0ull << taken) : 0ull;
#pragma unroll
                for (int u = 0; u < TEST; ++u) {
                    const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(in[u] >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((unsigned)in[u], 0));
                    if (__builtin_amdgcn_inverse_ballot_w64(in[u])) {
                        const int to = (tail + below) & (RING - 1);
                        const unsigned short key = (unsigned short)(16 * (buf + j0 + u * TK_WAVE + lane));
                        ring[to] = key;
                        if (to < CHUNK)
                            ring[RING + to] = key;
                    }
                    tail += __builtin_popcountll(in[u]);
                }
            } else if (!idle && stage0 + cnt > tail) {
                tail = stage0 + cnt;
            }
            while (tail - head >= CHUNK)
                sweep(CHUNK);
        }
        if (st + 1 < nstages) {
            // The next stage replaces the previous one in LDS: whatever is still to be swept or pending
            // from it comes first (the queue is in key order, so its head tells).
            if (head < before)
                sweep(tail - head);
            // (no chunk begins more than a stage before or behind `before`)
            while (__builtin_amdgcn_ballot_w64(qlen > 0 && ((b0 - before) & STAGE) != 0) != 0) {
                stale = moved = true;
                service();
            }
            before = tail;
            __syncthreads();  // every wave is done with the previous stage
            stash((st + 1) & 1);
        }
        __syncthreads();
    }
    if (tail > head)
        sweep(tail - head);
    while (__builtin_amdgcn_ballot_w64(qlen > 0) != 0)
        service();

    // ---- results: the workgroup's queries own consecutive rows of k; the slots go to their rows
    // through LDS (row stride KMAX + 1), a part of the rows at a time, so that the stores are runs
    // of consecutive elements ----
    float *const tbuf = skey;  // values, then indices
    int *const ibuf = reinterpret_cast<int *>(skey + ROWS * ROW);
#pragma unroll 1
    for (int part = 0; part < BLOCK / ROWS; ++part) {
        const int row0 = base + part * ROWS;  // of the cloud's queries
        int rows = (n1 - base < span ? n1 - base : span) - part * ROWS;
        if (rows <= 0)  // uniform
            break;
        rows = rows < ROWS ? rows : ROWS;
        __syncthreads();  // the last stage, or the part before, has been read
        if (active && mine / ROWS == part) {
            const int r = (mine & (ROWS - 1)) * ROW;
#pragma unroll
            for (int p = 0; p < KMAX; ++p) {
                if (p < k) {  // uniform
                    if constexpr (KMAX > 16)
                        asm volatile("" : "+v"(v[p]));  // (and the slots' addresses, ahead of the parts)
                    const int slot = Slot::slot(v[p]);
                    tbuf[r + slot] = __builtin_bit_cast(float, Slot::distance(v[p]));
                    ibuf[r + slot] = (int)(Slot::low(v[p]) & Slot::KEY);
                }
            }
            if (nan_slots != 0u) {  // NaNs of the fill, still in their slots
#pragma unroll
                for (int s = 0; s < KMAX; ++s) {
                    if (s < k && ((nan_slots >> s) & 1u))
                        tbuf[r + s] = tk_dist2<float>(knn_coord<SOA>(K, n2, s, 0), knn_coord<SOA>(K, n2, s, 1),
                                                      knn_coord<SOA>(K, n2, s, 2), qx, qy, qz);
                }
            }
        }
        __syncthreads();
        const int total = rows * k;
        float *od = distance + ((int64_t)b * n1 + row0) * k;
        int64_t *oi = index + ((int64_t)b * n1 + row0) * k;
        int r = tid / k, col = tid - r * k;
        const int dr = BLOCK / k, dcol = BLOCK - dr * k;
#pragma unroll 1
        for (int e = tid; e < total; e += BLOCK) {
            od[e] = tbuf[r * ROW + col];
            oi[e] = (int64_t)ibuf[r * ROW + col];
            r += dr;
            col += dcol;
            r += col >= k ? 1 : 0;
            col -= col >= k ? k : 0;
        }
        if constexpr (WEIGHTS) {  // k == 3
            for (int i = tid; i < rows; i += BLOCK) {
                const float d3[3] = {tbuf[i * ROW], tbuf[i * ROW + 1], tbuf[i * ROW + 2]};
                knn_three_weights<float>(d3, eps, weight + ((int64_t)b * n1 + row0 + i) * 3);
            }
        }
    }
}

template <int KMAX, bool SOA, bool WEIGHTS, int LANES, int KIND>
__global__ __launch_bounds__(LANES) void knn_filter_kernel_f32(
    const float *__restrict__ query, const float *__restrict__ key,
    float *__restrict__ distance, int64_t *__restrict__ index, float *__restrict__ weight,
    float eps, int blocks_per_batch, int n1, int n2, int k)
{
    using F = KnnFilter<KMAX, LANES>;
    constexpr int BLOCK = F::BLOCK, NW = F::NW, CELLS = F::CELLS;
    constexpr bool BOXES = KIND != KNN_EVERY_KEY, ORDERED = KIND == KNN_BOXES_UNLESS_ORDERED;
    __shared__ __align__(16) float skey[F::LDS_FLOATS];
    // (a list's beginning comes once more behind it)
    __shared__ __align__(16) unsigned short srings[BOXES ? NW * (F::RING + F::CHUNK) : 1];
    __shared__ float sred[NW][F::RED];
    const int tid = threadIdx.x;
    const int lane = tid & (TK_WAVE - 1);
    const int wave = tid / TK_WAVE;
    const bool second = ORDERED && blockIdx.y > 0;
    const int b = blockIdx.x / blocks_per_batch;
    const int qblock = blockIdx.x - b * blocks_per_batch;
    const float *__restrict__ K = key + (int64_t)b * n2 * 3;
    const float *__restrict__ Q = query + (int64_t)b * n1 * 3;
    const float INF = __builtin_huge_valf();

    // ---- bounding boxes of the key cloud (its centre, and a bound of the centred norms) and of the
    // workgroup's queries ----
    const int base = qblock * BLOCK;
    float ends[6] = {-INF, -INF, -INF, -INF, -INF, -INF};  // -lowest, highest
    for (int j = tid; j < n2; j += BLOCK) {
        const float v[3] = {knn_coord<SOA>(K, n2, j, 0), knn_coord<SOA>(K, n2, j, 1), knn_coord<SOA>(K, n2, j, 2)};
        knn_reach_out(ends, v);
    }
    KnnFrame<F::PER> frame;
    knn_filter_fetch<SOA, F::PER, BLOCK>(frame.pre, K, n2, 0);
    float qends[6] = {-INF, -INF, -INF, -INF, -INF, -INF};
#pragma unroll
    for (int a = 0; a < 3; ++a)
        frame.own[a] = 0.0f;  // (of a query that does not exist)
    if (BOXES && base + tid < n1) {
#pragma unroll
        for (int a = 0; a < 3; ++a)
            frame.own[a] = knn_coord<SOA>(Q, n1, base + tid, a);
        knn_reach_out(qends, frame.own);
    }
    const auto box_of_wave = [&](float (&e)[6], int at) {
        tk_wave_max_six<64>(e);
        if (lane == TK_WAVE - 1) {
#pragma unroll
            for (int a = 0; a < 6; ++a)
                sred[wave][at + a] = e[a];
        }
    };
    box_of_wave(ends, 0);
    if constexpr (BOXES)
        box_of_wave(qends, 6);
    if constexpr (ORDERED) {
        float first[6] = {-INF, -INF, -INF, -INF, -INF, -INF};  // of the first stage's keys
        if (tid < n2) {
            const float v[3] = {frame.pre[0].x, frame.pre[0].y, frame.pre[0].z};
            knn_reach_out(first, v);
        }
        box_of_wave(first, 12);
    }
    if constexpr (BOXES) {  // the sort's counters and its table
        unsigned *const cnt = reinterpret_cast<unsigned *>(skey);
        unsigned short *const curve = reinterpret_cast<unsigned short *>(cnt + CELLS + 4);
        if (tid < CELLS / 8)
            reinterpret_cast<uint4 *>(curve)[tid] = reinterpret_cast<const uint4 *>(knn_curve.place)[tid];
        for (int i = tid; i <= CELLS; i += BLOCK)
            cnt[i] = 0u;
    }
    __syncthreads();
    // (a wave's values to a lane: read one after the other they took more than the reductions in the waves)
    float all[6], queries[6], firsts[6];
    const auto box_of_all = [&](float (&e)[6], int at) {
#pragma unroll
        for (int a = 0; a < 6; ++a)
            e[a] = sred[lane & (NW - 1)][at + a];
        tk_wave_max_six<8>(e);
#pragma unroll
        for (int a = 0; a < 6; ++a)
            e[a] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e[a]), 7));
    };
    box_of_all(all, 0);
    if constexpr (BOXES)
        box_of_all(queries, 6);
    if constexpr (ORDERED)
        box_of_all(firsts, 12);
    float kmax2 = 0.0f;
    bool ordered = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float l = all[a], h = all[3 + a];
        if (ORDERED)
            ordered = ordered || firsts[3 + a] + firsts[a] < 0.6f * (h + l);
        const float middle = 0.5f * h - 0.5f * l, side = __builtin_fmaxf(h - middle, middle + l);
        frame.centre[a] = middle;
        // (the operations of a norm, each of which is monotone: no centred key is beyond it)
        kmax2 = a == 0 ? side * side : __builtin_fmaf(side, side, kmax2);
        if (BOXES) {
            frame.origin[a] = -queries[a];
            const float extent = queries[3 + a] + queries[a];
            frame.cells[a] = extent > 0.0f ? 7.99f / extent : 0.0f;  // also 0 for NaN / inf extents
        }
    }
    const float c0 = frame.centre[0], c1 = frame.centre[1], c2 = frame.centre[2];
    bool safe = (c0 - c0 == 0.0f) && (c1 - c1 == 0.0f) && (c2 - c2 == 0.0f) && (kmax2 < 1e30f);
    const float ext = __builtin_sqrtf(kmax2);
    const int ebits = (int)((__builtin_bit_cast(unsigned, ext) >> 23) & 0xffu) - 127;
    safe = safe && (ext == 0.0f || (ebits >= -40 && ebits <= 40));
    // Half the box's diagonal comes to [2, 4): its largest side is 1/sqrt(3) of that or more, and a key on it.
    frame.scale = (!safe || ext == 0.0f) ? 1.0f : __builtin_bit_cast(float, (unsigned)(128 - ebits) << 23);
    frame.kmax = __builtin_sqrtf(kmax2) * frame.scale * 1.000001f;

    // (the same in all lanes, which the compiler cannot know)
    const bool every = !BOXES || (ORDERED && __builtin_amdgcn_readfirstlane(ordered) != 0);
    if (__builtin_amdgcn_readfirstlane(!safe || (second && !every))) {
        if (!second)
            knn_batched_body<KMAX, SOA, WEIGHTS>(query, key, distance, index, weight, eps, b, base + tid, n1, n2, k,
                                                 skey);
        return;
    }
    const auto run = [&](auto boxes, int from, int span) {
        knn_filter_queries<KMAX, SOA, WEIGHTS, LANES, decltype(boxes)::value>(Q, K, distance, index, weight, eps, b, from,
                                                                              span, n1, n2, k, frame, skey, srings, sred);
    };
    if constexpr (KIND == KNN_EVERY_KEY) {
        run(std::false_type{}, base, BLOCK);
    } else if constexpr (KIND == KNN_BOXES) {
        run(std::true_type{}, base, BLOCK);
    } else {
        if (!every)
            run(std::true_type{}, base, BLOCK);
        else
            run(std::false_type{}, second ? base + BLOCK / 2 : base, gridDim.y > 1 ? BLOCK / 2 : BLOCK);
    }
}


// fp32 variant with the slots in LDS as a per-lane tournament tree.
//
// With the slots in registers every insertion pays O(k) selects and compares, because
// registers cannot be indexed per lane. LDS can: a lane keeps, in columns of its own
// (row r of an array at [r * 64 + lane], conflict-free whatever r each lane uses),
//   leaf[s]  distance in slot s           kidx[s]  key index in slot s
//   ival[n]  largest distance below node n of a binary tree over the slots (heap
//            numbering, node 1 the root, the leaf of slot s at KMAX + s)
//   iarg[n]  the first slot that holds ival[n]
// ival / iarg exist for nodes 1 .. KMAX/2-1 only: a parent of two leaves is worked out
// from its leaves when needed, which saves a quarter of the LDS (the LDS footprint
// decides how many waves a CU holds). An insertion overwrites the leaf of the current
// maximum and replays the log2(KMAX) matches on the way to the root. The other side of
// each of those matches is known up front, so all of them are fetched at once and the
// path costs one LDS round trip plus three vector instructions per level. A right child
// wins a match only when strictly greater, so a node reports the first slot holding its
// maximum - MinK's rescan order (mink.cuh:74-87); MinK starts that rescan from the
// inserted key, hence the maximum stays in the inserted slot when the root is not
// strictly above it.
//
// The sweep takes its keys through scalar loads (the address is the same for every
// lane) and the rounds fetch their candidates straight from global memory, one round
// ahead; a block is one wave and never synchronises. IDX16 stores key indices in 16
// bits (clouds up to 65536 keys).
//
// NaN distances can only enter during the fill (a later key must compare below the
// maximum). MinK never selects such a slot as maximum unless it is slot 0, in which
// case it never inserts again. Here a NaN in slot 0 freezes the lane; a NaN elsewhere
// plays the tournament as -inf and is recomputed when the results are written.
template <int KMAX, bool IDX16, typename T = float> struct KnnTreeLayout {
    static constexpr int NT = 64;
    using Idx = typename std::conditional<IDX16, unsigned short, int>::type;
    static constexpr int LEAF_BYTES = (int)sizeof(T) * KMAX * NT;
    static constexpr int KIDX_BYTES = (int)sizeof(Idx) * KMAX * NT;
    static constexpr int IVAL_BYTES = (int)sizeof(T) * (KMAX / 2) * NT;
    static constexpr int IARG_BYTES = (KMAX / 2) * NT;
    static constexpr int BYTES = LEAF_BYTES + KIDX_BYTES + IVAL_BYTES + IARG_BYTES;
};

template <typename T, int KMAX, bool IDX16, bool SOA = false>
__global__ __launch_bounds__(64) void knn_tree_kernel(
    const T *__restrict__ query, const T *__restrict__ key,
    T *__restrict__ distance, int64_t *__restrict__ index, int blocks_per_batch, int n1,
    int n2, int k)
{
    using Lay = KnnTreeLayout<KMAX, IDX16, T>;
    using Idx = typename Lay::Idx;
    constexpr int CHUNK = 32;
    constexpr int NT = 64;
    constexpr int HALF = KMAX / 2;  // nodes HALF .. KMAX-1 are the parents of the leaves
    constexpr int LEVELS = KMAX == 8 ? 3 : KMAX == 16 ? 4 : KMAX == 32 ? 5 : KMAX == 64 ? 6
                           : KMAX == 128 ? 7 : 8;
    static_assert((1 << LEVELS) == KMAX, "KMAX must be a power of two from 8 to 256");
    static_assert(KMAX <= 256, "slot numbers are kept in one byte");
    extern __shared__ __align__(16) unsigned char knn_tree_lds[];
    const int lane = threadIdx.x;
    T *const leaf = reinterpret_cast<T *>(knn_tree_lds) + lane;
    Idx *const kidx = reinterpret_cast<Idx *>(knn_tree_lds + Lay::LEAF_BYTES) + lane;
    T *const ival =
        reinterpret_cast<T *>(knn_tree_lds + Lay::LEAF_BYTES + Lay::KIDX_BYTES) + lane;
    unsigned char *const iarg =
        knn_tree_lds + Lay::LEAF_BYTES + Lay::KIDX_BYTES + Lay::IVAL_BYTES + lane;

    const int b = blockIdx.x / blocks_per_batch;
    const int qi = (blockIdx.x - b * blocks_per_batch) * NT + lane;
    const bool active = qi < n1;
    const T *__restrict__ K = key + (int64_t)b * n2 * 3;
    T qx = 0, qy = 0, qz = 0;
    if (active) {
        const T *__restrict__ Q = query + (int64_t)b * n1 * 3;
        qx = knn_coord<SOA>(Q, n1, qi, 0);
        qy = knn_coord<SOA>(Q, n1, qi, 1);
        qz = knn_coord<SOA>(Q, n1, qi, 2);
    }

    // Value and first slot of a node whose children are leaves.
    auto leaf_parent = [&](int n, T &v, int &a) {
        const int s = 2 * n - KMAX;
        const T lv = leaf[s * NT], rv = leaf[(s + 1) * NT];
        const bool right = rv > lv;
        v = right ? rv : lv;
        a = right ? s + 1 : s;
    };

    // Fill phase: keys 0..k-1 go to slots 0..k-1 (mink.cuh:63-72); unused slots hold -inf.
    bool frozen = false;
    for (int s = 0; s < KMAX; ++s) {
        T d = -tk_inf<T>();
        if (s < k) {
            d = tk_dist2<T>(knn_coord<SOA>(K, n2, s, 0), knn_coord<SOA>(K, n2, s, 1),
                                knn_coord<SOA>(K, n2, s, 2), qx, qy, qz);
            if (d != d) {
                frozen |= s == 0;
                d = -tk_inf<T>();  // marks the slot: no real distance is -inf
            }
        }
        leaf[s * NT] = d;
        kidx[s * NT] = (Idx)s;
    }
    for (int n = HALF - 1; n >= 1; --n) {
        T lv, rv;
        int la, ra;
        if (2 * n >= HALF) {
            leaf_parent(2 * n, lv, la);
            leaf_parent(2 * n + 1, rv, ra);
        } else {
            lv = ival[2 * n * NT];
            rv = ival[(2 * n + 1) * NT];
            la = iarg[2 * n * NT];
            ra = iarg[(2 * n + 1) * NT];
        }
        const bool right = rv > lv;
        ival[n * NT] = right ? rv : lv;
        iarg[n * NT] = (unsigned char)(right ? ra : la);
    }
    T max_key = frozen ? -tk_inf<T>() : ival[NT];
    int max_idx = iarg[NT];

    for (int first = 0; first < n2; first += CHUNK) {  // `first` = key index of bit 31
        // ---- sweep: bit (31 - i) of `mask` <=> key first+i is below the maximum ----
        // (fp32: squared distances are non-negative, their bit patterns order as integers
        // and the sign of the difference is shifted in with one instruction)
        auto below_max = [&](unsigned m, T d) {
            if constexpr (sizeof(T) == 4) {
                const unsigned diff = (unsigned)(__builtin_bit_cast(int, d) -
                                                 __builtin_bit_cast(int, max_key));
                return __builtin_amdgcn_alignbit(m, diff, 31);  // (m << 1) | sign
            } else {
                return (m << 1) | (d < max_key ? 1u : 0u);
            }
        };
        unsigned mask = 0u;
        if (first + CHUNK <= n2) {
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) {  // (wave-uniform addresses: scalar loads)
                const T d = tk_dist2<T>(knn_coord<SOA>(K, n2, first + i, 0),
                                        knn_coord<SOA>(K, n2, first + i, 1),
                                        knn_coord<SOA>(K, n2, first + i, 2), qx, qy, qz);
                mask = below_max(mask, d);
            }
        } else {
            for (int i = 0; i < CHUNK; ++i) {
                const int j = first + i < n2 ? first + i : n2 - 1;  // clamped, masked below
                const T d = tk_dist2<T>(knn_coord<SOA>(K, n2, j, 0), knn_coord<SOA>(K, n2, j, 1),
                                        knn_coord<SOA>(K, n2, j, 2), qx, qy, qz);
                mask = below_max(mask, d);
            }
        }
        // Keys that do not exist, or that the fill phase took, are no candidates.
        int lo = k - first;                          // keys below k filled the slots
        lo = lo < 0 ? 0 : (lo > CHUNK ? CHUNK : lo);
        int hi = n2 - first;                         // keys at or beyond hi do not exist
        hi = hi > CHUNK ? CHUNK : hi;
        unsigned valid = (lo >= CHUNK) ? 0u : (0xffffffffu >> lo);
        valid &= (hi >= CHUNK) ? 0xffffffffu : ~(0xffffffffu >> hi);
        mask &= valid;

        // ---- insertion rounds, the next candidate's key in flight during the current ----
        bool has = mask != 0u;
        int i = has ? __builtin_clz(mask) : 0;
        T ex = knn_coord<SOA>(K, n2, first + i, 0), ey = knn_coord<SOA>(K, n2, first + i, 1),
          ez = knn_coord<SOA>(K, n2, first + i, 2);
        while (__builtin_amdgcn_ballot_w64(has)) {  // wave-uniform
            mask &= ~(0x80000000u >> i);  // no-op for a lane without a candidate
            const bool has_next = mask != 0u;
            const int i_next = has_next ? __builtin_clz(mask) : 0;
            const T nx = knn_coord<SOA>(K, n2, first + i_next, 0),
                    ny = knn_coord<SOA>(K, n2, first + i_next, 1),
                    nz = knn_coord<SOA>(K, n2, first + i_next, 2);
            const T d = tk_dist2<T>(ex, ey, ez, qx, qy, qz);
            if (has && d < max_key) {
                const int p = max_idx;
                leaf[p * NT] = d;
                kidx[p * NT] = (Idx)(first + i);
                // the other side of every match on the path, fetched together
                T sv[LEVELS];
                int sa[LEVELS];
                sv[0] = leaf[(p ^ 1) * NT];
                sa[0] = p ^ 1;
                leaf_parent(((KMAX + p) >> 1) ^ 1, sv[1], sa[1]);
#pragma unroll
                for (int l = 2; l < LEVELS; ++l) {
                    const int sib = ((KMAX + p) >> l) ^ 1;
                    sv[l] = ival[sib * NT];
                    sa[l] = iarg[sib * NT];
                }
                T v = d;
                int a = p;
#pragma unroll
                for (int l = 0; l < LEVELS; ++l) {
                    const int node = (KMAX + p) >> l;
                    // the other side wins from the right only when strictly greater
                    const bool take = (node & 1) ? !(v > sv[l]) : (sv[l] > v);
                    v = take ? sv[l] : v;
                    a = take ? sa[l] : a;
                    // parents of leaves are not stored; the root lives in max_key / max_idx
                    if (l >= 1 && l + 1 < LEVELS) {
                        ival[(node >> 1) * NT] = v;
                        iarg[(node >> 1) * NT] = (unsigned char)a;
                    }
                }
                max_key = v;
                max_idx = v != d ? a : p;
            }
            has = has_next;
            i = i_next;
            ex = nx;
            ey = ny;
            ez = nz;
        }
    }

    if (active) {
        T *od = distance + ((int64_t)b * n1 + qi) * k;
        int64_t *oi = index + ((int64_t)b * n1 + qi) * k;
        for (int s = 0; s < k; ++s) {
            T d = leaf[s * NT];
            if (d == -tk_inf<T>())  // a NaN of the fill phase, still in its slot
                d = tk_dist2<T>(knn_coord<SOA>(K, n2, s, 0), knn_coord<SOA>(K, n2, s, 1),
                                knn_coord<SOA>(K, n2, s, 2), qx, qy, qz);
            od[s] = d;
            oi[s] = (int64_t)kidx[s * NT];
        }
    }
}

template <int KMAX, bool IDX16, typename T = float, bool SOA = false>
int knn_tree_launch_as(const T *query, const T *key, T *distance, int64_t *index,
                       int64_t B, int n1, int n2, int k, hipStream_t s)
{
    constexpr int LDS_BYTES = KnnTreeLayout<KMAX, IDX16, T>::BYTES;
    if (LDS_BYTES > 48 * 1024) {
        const int allowed =
            tk_allow_dynamic_lds<knn_tree_kernel<T, KMAX, IDX16, SOA>>(LDS_BYTES);
        if (allowed != TK3D_OK)
            return allowed;
    }
    const int64_t bpb = ((int64_t)n1 + 63) / 64;
    if (B * bpb > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((knn_tree_kernel<T, KMAX, IDX16, SOA>), dim3((unsigned)(B * bpb)), dim3(64),
                       LDS_BYTES, s, query, key, distance, index, (int)bpb, n1, n2, k);
    return tk_launch_status();
}

template <int KMAX, typename T = float, bool SOA = false>
int knn_tree_launch(const T *query, const T *key, T *distance, int64_t *index,
                    int64_t B, int n1, int n2, int k, hipStream_t s)
{
    if (n2 <= 65536)
        return knn_tree_launch_as<KMAX, true, T, SOA>(query, key, distance, index, B, n1, n2, k, s);
    return knn_tree_launch_as<KMAX, false, T, SOA>(query, key, distance, index, B, n1, n2, k, s);
}

// ---- a wave per query ---------------------------------------------------------------------------
//
// With a lane per query a launch needs 65536 queries to give every SIMD a wave, and an insertion
// is a chain of dependent LDS or register steps for the whole wave. Here a wave has ONE query and
// up to 64 slots, one per lane: 64 keys are measured at once, and those below the maximum are
// inserted one after the other in key order, which are MinK's insertions in MinK's order. The
// kernel is bound by the chain of an insertion, about k (1 + ln(N2 / k)) times per query in random key
// order. The lanes hold the slots in descending order, as the doubles of the kernel above
// (distance, flag, slot, key; KnnSlot): the head leaves, and a lane takes the larger of its lower
// neighbour's and the smaller of its own and the new key's - two moves between lanes, a minimum and a
// maximum, where slots that stay in their lanes take two selects and a maximum over the lanes (4, 5 or
// 6 steps). A list of the lanes that moves distance, slot and key by selects was slower than either.
// us, slots that stay in their lanes and now: 4 x 512 queries on 16384 keys k = 16 39.2, 33.3, k = 64 70.6, 54.4; 1 x
// 4096 on 16384 k = 64 93, 76; 8 x 2048 on 4096 k = 20 79, 68, k = 64 159, 124; on short clouds, where ordering the
// first k counts, 8 x 2048 on 128 k = 64 27.6, 23.9, on 64 k = 32 16.4, 14.3. Tried: insertions in a row
// without a look at the new maximum (longer for few neighbours, whose maximum falls fast).
// A NaN of the fill holds the pattern of -inf, below every distance; one in slot 0 freezes the query,
// and no comparison takes one as a candidate.

// The value of lane (l ^ X) for X below 32, or 63.
template <int X> __device__ __forceinline__ int knn_lane_xor(int v)
{
    constexpr int DPP = X == 1 ? 0xb1 : X == 2 ? 0x4e : X == 3 ? 0x1b  // quad_perm
                        : X == 7 ? 0x141 : X == 15 ? 0x140             // row_half_mirror, row_mirror
                        : X == 8 ? 0x128 : 0;                          // row_ror:8
    if constexpr (DPP != 0)
        return __builtin_amdgcn_mov_dpp(v, DPP, 0xf, 0xf, true);
    else if constexpr (X < 32)
        return __builtin_amdgcn_ds_swizzle(v, (X << 10) | 0x1f);
    else
        return __shfl_xor(v, X);
}

// A step of the network below: the lower lane of a pair l, l ^ X keeps the larger double.
template <int X> __device__ __forceinline__ void knn_order_step(int &vh, int &vl, int lane)
{
    const int oh = knn_lane_xor<X>(vh), ol = knn_lane_xor<X>(vl);
    const bool lower = (lane & (X == 63 ? 32 : X == 31 ? 16 : X == 15 ? 8 : X == 7 ? 4 : X == 3 ? 2 : X)) == 0;
    const double mine = __builtin_bit_cast(double, (unsigned long long)(unsigned)vh << 32 | (unsigned)vl);
    const double other = __builtin_bit_cast(double, (unsigned long long)(unsigned)oh << 32 | (unsigned)ol);
    const bool take = (other > mine) == lower;
    vh = take ? oh : vh;
    vl = take ? ol : vl;
}

// The doubles of the first k lanes in descending order, -inf in the others: a bitonic network of 1, 3, 6, 10, 15 or
// 21 steps, of the size that holds k lanes. (Counting, for every lane, the values above its own took four instructions
// a value: 8 x 2048 queries on 128 keys, k = 64 30.4 us, 23.9 now.)
__device__ __forceinline__ void knn_order_lanes(int &vh, int &vl, int lane, int k)
{
    if (k > 1)  // (uniform)
        knn_order_step<1>(vh, vl, lane);
    if (k > 2) {
        knn_order_step<3>(vh, vl, lane);
        knn_order_step<1>(vh, vl, lane);
    }
    if (k > 4) {
        knn_order_step<7>(vh, vl, lane);
        knn_order_step<2>(vh, vl, lane);
        knn_order_step<1>(vh, vl, lane);
    }
    if (k > 8) {
        knn_order_step<15>(vh, vl, lane);
        knn_order_step<4>(vh, vl, lane);
        knn_order_step<2>(vh, vl, lane);
        knn_order_step<1>(vh, vl, lane);
    }
    if (k > 16) {
        knn_order_step<31>(vh, vl, lane);
        knn_order_step<8>(vh, vl, lane);
        knn_order_step<4>(vh, vl, lane);
        knn_order_step<2>(vh, vl, lane);
        knn_order_step<1>(vh, vl, lane);
    }
    if (k > 32) {
        knn_order_step<63>(vh, vl, lane);
        knn_order_step<16>(vh, vl, lane);
        knn_order_step<8>(vh, vl, lane);
        knn_order_step<4>(vh, vl, lane);
        knn_order_step<2>(vh, vl, lane);
        knn_order_step<1>(vh, vl, lane);
    }
}

// CHUNKS: of 64 keys each, requested together, eight or as many as a short cloud has (8 x 2048 queries on 64 keys, k =
// 3: 10.2 us with eight, 8.5 with one). LONG: clouds of more than KNN_SLOT_KEYS keys, whose numbers do not fit beside a
// slot and go along in a register of their own (16 queries on 2^25 + 4096 keys, k = 32, by the kernel of a lane per
// query 487 ms, here 44; k = 64, with slots in a tree in LDS, 2870 and 45).
constexpr int KNN_SLOT_KEYS = 1 << 25;

// A trip inside the cloud loads from uniform addresses at the lane's offset and asks about no key whether it exists or
// was filled (17 vector instructions a chunk, one of them a product of integers, became 8), and 64 registers leave room for eight
// waves a SIMD (67 before). us, before and now: 4 x 512 queries on 10000 keys k = 1 16.6, 14.2, k = 64 45.4, 42.4; 8 x
// 2048 on 2048 k = 20 50, 45; 1 x 16384 on 16384 k = 3 123, 119 (its loads from L1), k = 16 163, 140, k = 64 232, 183; planes, 1 x
// 16384 on 4096 k = 3 43.7, 36.3; one trip, 8 x 2048 on 300 k = 16 24.9, 23.9.
template <int CHUNKS, bool LONG, bool SOA, bool WEIGHTS>
__global__ __launch_bounds__(KNN_BLOCK, LONG ? 1 : 8) void knn_wave_kernel_f32(
    const float *__restrict__ query, const float *__restrict__ key, float *__restrict__ distance,
    int64_t *__restrict__ index, float *__restrict__ weight, float eps, int64_t queries, int n1,
    int n2, int k, int sorted, int root)
{
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (KNN_BLOCK / 64) +
                        __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= queries)
        return;
    const int b = (int)(row / n1), qi = (int)(row - (int64_t)b * n1);
    const float *__restrict__ Q = query + (int64_t)b * n1 * 3;
    const float *__restrict__ K = key + (int64_t)b * n2 * 3;
    const float qx = knn_coord<SOA>(Q, n1, qi, 0), qy = knn_coord<SOA>(Q, n1, qi, 1),
                qz = knn_coord<SOA>(Q, n1, qi, 2);

    float px[CHUNKS], py[CHUNKS], pz[CHUNKS];
    constexpr int TRIP = 64 * CHUNKS;
    const unsigned lane_bytes = (unsigned)lane * (SOA ? 4u : 12u);
    const auto load = [&](int base) {
        if (CHUNKS == 8 && base > 0 && base + TRIP <= n2) {  // uniform: a lane's offset to uniform addresses
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c) {
                const char *const at = reinterpret_cast<const char *>(K + (int64_t)(base + 64 * c) * (SOA ? 1 : 3));
                if constexpr (SOA) {
                    px[c] = *reinterpret_cast<const float *>(at + lane_bytes);
                    py[c] = *reinterpret_cast<const float *>(at + (int64_t)n2 * 4 + lane_bytes);
                    pz[c] = *reinterpret_cast<const float *>(at + (int64_t)n2 * 8 + lane_bytes);
                } else {
                    const TkPoint3<float> p = *reinterpret_cast<const TkPoint3<float> *>(at + lane_bytes);
                    px[c] = p.x;
                    py[c] = p.y;
                    pz[c] = p.z;
                }
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            int j = base + 64 * c + lane;
            j = j < n2 ? j : n2 - 1;
            if constexpr (SOA) {
                px[c] = K[j];
                py[c] = K[n2 + j];
                pz[c] = K[2 * n2 + j];
            } else {
                // (a 32-bit offset to a uniform address, if it fits)
                using Offset = typename std::conditional<LONG, int64_t, unsigned>::type;
                const TkPoint3<float> p = *reinterpret_cast<const TkPoint3<float> *>(
                    reinterpret_cast<const char *>(K) + (Offset)j * 12);
                px[c] = p.x;
                py[c] = p.y;
                pz[c] = p.z;
            }
        }
    };
    load(0);

    using Slot = KnnSlot<64>;
    // The first k keys fill the slots (mink.cuh:63-72): key s in slot s, put in order here. With a
    // NaN in slot 0 MinK's maximum is a NaN, which nothing is below.
    const float filled = tk_dist2<float>(px[0], py[0], pz[0], qx, qy, qz);
    const bool nan = filled != filled;
    constexpr int UNUSED = (int)0xfff00000u;  // a double's -inf, below all others
    int vh = lane >= k ? UNUSED : nan ? (int)0xff800000u : __float_as_int(filled);
    int vl = lane >= k ? 0 : (63 - lane) << Slot::KEY_BITS;
    if constexpr (!LONG)
        vl |= lane >= k ? 0 : lane;
    if (k < n2 || sorted)  // (else nothing leaves, and every key goes to its slot)
        knn_order_lanes(vh, vl, lane, k);
    const auto slot_of = [](int low) { return 63 - (int)(((unsigned)low & Slot::SLOT) >> Slot::KEY_BITS); };
    int vk = LONG ? slot_of(vl) : 0;
    const bool frozen = __builtin_amdgcn_readfirstlane((int)nan) != 0;
    // what a key has to be below
    unsigned top = (unsigned)__builtin_amdgcn_readfirstlane(vh);
    top = frozen || (int)top < 0 ? 0u : top;

    for (int base = 0; base < n2; base += TRIP) {
        unsigned d[CHUNKS];
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
            d[c] = __float_as_uint(tk_dist2<float>(px[c], py[c], pz[c], qx, qy, qz));
        if (base == 0 || base + TRIP > n2) {  // uniform
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c) {
                const int j = base + 64 * c + lane;
                d[c] = j >= k && j < n2 ? d[c] : 0xffffffffu;
            }
        }
        if (base + TRIP < n2)
            load(base + TRIP);
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            unsigned long long mask = __ballot(d[c] < top);
            while (mask) {
                const int l = (int)__builtin_ctzll(mask);
                const int xh = __builtin_amdgcn_readlane((int)d[c], l);
                // the slot of the maximum, which leaves; with nothing that stays strictly above it
                // the key goes to the head, also in front of its equals (mink.cuh:74-87)
                const unsigned slot = (unsigned)__builtin_amdgcn_readfirstlane(vl) & Slot::SLOT;
                const unsigned flag = xh >= __builtin_amdgcn_readlane(vh, 1) ? Slot::FLAG : 0u;
                const int number = base + 64 * c + l;
                const double x = Slot::pack(xh, slot | flag | (LONG ? 0u : (unsigned)number));
                const double mine = Slot::pack(vh, (unsigned)vl);
                const double next = Slot::pack(
                    __builtin_amdgcn_update_dpp(UNUSED, vh, 0x130, 0xf, 0xf, false),  // wave_shl:1
                    (unsigned)__builtin_amdgcn_update_dpp(0, vl, 0x130, 0xf, 0xf, true));
                const double v = knn_max_f64(next, knn_min_f64_uniform(mine, x));
                if constexpr (LONG) {  // (no two slots are equal: v is one of the three)
                    const int below = __builtin_amdgcn_update_dpp(0, vk, 0x130, 0xf, 0xf, true);
                    vk = v == next ? below : v == mine ? vk : number;
                }
                vh = Slot::distance(v);
                vl = (int)Slot::low(v);
                top = (unsigned)__builtin_amdgcn_readfirstlane(vh);
                mask = __ballot(d[c] < top) & (~1ull << l);
            }
        }
    }

    // An entry goes to its slot, or to its place in ascending order (equal distances in slot
    // order, NaNs last, as a stable sort of the slots leaves them).
    const int slot = slot_of(vl);
    const float refilled = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * slot, __float_as_int(filled)));
    float out = vh < 0 ? refilled : __int_as_float(vh);  // (a NaN never leaves its slot)
    int place = slot;
    if (sorted) {
        // equal neighbours, or NaNs: counted
        const int below = __builtin_amdgcn_update_dpp(UNUSED, vh, 0x130, 0xf, 0xf, false);
        place = k - 1 - lane;
        if (__ballot(lane < k && (vh < 0 || vh == below))) {
            place = 0;
            for (int l = 0; l < k; ++l) {
                const unsigned other = (unsigned)__builtin_amdgcn_readlane(vh, l);  // (NaN: the largest)
                const int there = __builtin_amdgcn_readlane(slot, l);
                place += other < (unsigned)vh || (other == (unsigned)vh && there < slot) ? 1 : 0;
            }
        }
    }
    if (root)
        out = __builtin_sqrtf(out);
    if (lane < k) {
        distance[row * k + place] = out;
        index[row * k + place] = LONG ? (int64_t)vk : (int64_t)((unsigned)vl & Slot::KEY);
    }
    if constexpr (WEIGHTS) {  // k == 3
        const int of_slot = __builtin_amdgcn_ds_permute(4 * (lane < k ? slot : lane), __float_as_int(out));
        float d3[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            d3[i] = __int_as_float(__builtin_amdgcn_readlane(of_slot, i));
        float w[3];
        knn_three_weights<float>(d3, eps, w);
        if (lane < 3)
            weight[row * 3 + lane] = lane == 0 ? w[0] : lane == 1 ? w[1] : w[2];
    }
}

// Up to how many queries a wave per query wins: its time goes with their number, that of the kernels of a lane per
// query hardly does while they leave CUs idle. Its time over that of the pre-filtered kernel, keys in random order
// and in that of a coordinate, clouds of 512 to 4096 queries:
//   queries       keys    64         512        1024       2048       4096       8192       16384
//   20480  k = 1       0.89 0.82  0.68 0.66  0.65 0.65  0.76 0.68  0.96 0.68  1.13 0.73  1.25 0.80
//          k = 3       1.07 1.08  0.89 0.92  0.80 0.86  0.74 0.90  0.88 0.90  1.03 0.88  1.18 0.84
//          k = 8       1.16 1.29  1.05 1.08  0.96 1.05  0.82 1.00  0.79 1.05  0.89 0.99  1.04 0.95
//          k = 16      1.10 1.22  1.06 0.95  0.99 0.95  0.88 0.92  0.75 0.89  0.72 0.94  0.88 0.89
//   24576  k = 1       1.03 0.91  0.79 0.75  0.75 0.73  0.90 0.76  1.12 0.78  1.36 0.85  1.48 0.94
//          k = 3       1.22 1.24  1.03 1.00  0.92 0.97  0.86 1.03  1.04 1.02  1.24 1.01  1.37 0.99
//          k = 8       1.34 1.44  1.20 1.21  1.11 1.18  0.95 1.12  0.92 1.19  1.07 1.14  1.26 1.09
//          k = 16      1.26 1.37  1.22 1.07  1.16 1.07  1.01 1.03  0.87 1.01  0.85 1.06  1.04 1.01
//          k = 32      0.92 0.96  0.96 0.85  0.98 0.85  0.92 0.82  0.83 0.82  0.74 0.79  0.69 0.76
//   32768  k = 1       1.25 1.13  0.95 0.93  0.94 0.91  1.15 0.97  1.48 1.00  1.79 1.07  1.99 1.23
//          k = 20      1.20 1.24  1.16 0.99  1.16 1.00  1.06 0.99  0.97 0.97  0.89 0.94  0.93 0.90
//          k = 32      1.17 1.19  1.22 1.06  1.26 1.06  1.17 1.03  1.06 1.03  0.98 0.99  0.89 0.95
// (on 65536, 32768 queries in clouds of 128 k = 20 1.06 1.29). With more than 32 neighbours the others keep a tree in
// LDS: us, the wave and the tree, 49152 queries on 128 keys k = 64 59, 72, on 4096 301, 549; 65536 on 1024 253, 243;
// 131072 on 128 k = 40 146, 136, on 4096 k = 40 570, 985, k = 64 771, 1143.
inline int64_t knn_wave_queries(int64_t keys, int64_t k)
{
    if (k > 32)
        return k > 64 ? 0 : keys >= 2048 ? 131072 : 49152;
    if (k > 16)
        return keys <= 1024 ? 25600 : keys <= 4096 ? 28672 : keys <= 32768 ? 32768 : 25600;
    if (keys <= 1024)
        return k <= 2 ? 30720 : k <= 4 || keys > 512 ? 20480 : 18432;
    if (keys <= 4096)
        return k > 4 && k <= 8 ? 23552 : 25600;
    return k > 8 && keys <= 8192 ? 25600 : 20480;
}
inline bool knn_wave_pays(int64_t queries, int64_t keys, int64_t k) { return queries <= knn_wave_queries(keys, k); }

template <bool SOA, bool WEIGHTS>
int knn_wave_launch(const float *query, const float *key, float *distance, int64_t *index,
                    float *weight, float eps, int64_t B, int n1, int n2, int k, int sorted,
                    int root, hipStream_t s)
{
    const int64_t queries = B * n1, blocks = (queries + KNN_BLOCK / 64 - 1) / (KNN_BLOCK / 64);
    if (k > 64 || blocks > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
#define TK_WAVE_LAUNCH(CHUNKS, LONG)                                                                             \
    hipLaunchKernelGGL((knn_wave_kernel_f32<CHUNKS, LONG, SOA, WEIGHTS>), dim3((unsigned)blocks), dim3(KNN_BLOCK), \
                       0, s, query, key, distance, index, weight, eps, queries, n1, n2, k, sorted, root)
    if (n2 <= 64)
        TK_WAVE_LAUNCH(1, false);
    else if (n2 <= 128)
        TK_WAVE_LAUNCH(2, false);
    else if (n2 <= 256)
        TK_WAVE_LAUNCH(4, false);
    else if (n2 <= KNN_SLOT_KEYS)
        TK_WAVE_LAUNCH(8, false);
    else
        TK_WAVE_LAUNCH(8, true);
#undef TK_WAVE_LAUNCH
    return tk_launch_status();
}

// Any k: the structure lives in the output rows in global memory.
template <typename T>
__global__ __launch_bounds__(KNN_BLOCK) void knn_global_kernel(
    const T *__restrict__ query, const T *__restrict__ key, T *distance, int64_t *index,
    int blocks_per_batch, int n1, int n2, int k)
{
    __shared__ T skey[KNN_STAGE * 4];
    const int tid = threadIdx.x;
    const int b = blockIdx.x / blocks_per_batch;
    const int qi = (blockIdx.x - b * blocks_per_batch) * KNN_BLOCK + tid;
    const bool active = qi < n1;
    const T *__restrict__ K = key + (int64_t)b * n2 * 3;
    T qx = 0, qy = 0, qz = 0;
    T *kd = distance;
    int64_t *ki = index;
    if (active) {
        const T *q = query + ((int64_t)b * n1 + qi) * 3;
        qx = q[0];
        qy = q[1];
        qz = q[2];
        kd = distance + ((int64_t)b * n1 + qi) * k;
        ki = index + ((int64_t)b * n1 + qi) * k;
    }
    T max_key = (T)0;
    int max_idx = 0;
    int size = 0;
    for (int stage0 = 0; stage0 < n2; stage0 += KNN_STAGE) {
        __syncthreads();
        for (int j = tid; j < KNN_STAGE; j += KNN_BLOCK) {
            const int kj = stage0 + j;
            T x = 0, y = 0, z = 0;
            if (kj < n2) {
                x = K[(int64_t)kj * 3 + 0];
                y = K[(int64_t)kj * 3 + 1];
                z = K[(int64_t)kj * 3 + 2];
            }
            skey[j * 4 + 0] = x;
            skey[j * 4 + 1] = y;
            skey[j * 4 + 2] = z;
            skey[j * 4 + 3] = (T)0;
        }
        __syncthreads();
        if (!active)
            continue;
        const int left = n2 - stage0;
        const int cnt = left < KNN_STAGE ? left : KNN_STAGE;
        for (int j = 0; j < cnt; ++j) {
            const T d = tk_dist2<T>(skey[j * 4 + 0], skey[j * 4 + 1], skey[j * 4 + 2], qx, qy,
                                    qz);
            const int kj = stage0 + j;
            if (size < k) {
                kd[size] = d;
                ki[size] = kj;
                if (size == 0 || d > max_key) {
                    max_key = d;
                    max_idx = size;
                }
                ++size;
            } else if (d < max_key) {
                kd[max_idx] = d;
                ki[max_idx] = kj;
                max_key = d;
                for (int s = 0; s < k; ++s) {
                    const T cur = kd[s];
                    if (cur > max_key) {
                        max_key = cur;
                        max_idx = s;
                    }
                }
            }
        }
    }
}

template <typename T, int KMAX, bool SOA = false, bool WEIGHTS = false>
void knn_launch(const T *query, const T *key, T *distance, int64_t *index, int64_t B,
                int bpb, int n1, int n2, int k, hipStream_t s, T *weight = nullptr,
                T eps = (T)0)
{
    if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((knn_batched_kernel_f32<KMAX, SOA, WEIGHTS>),
                           dim3((unsigned)(B * bpb)), dim3(KNN_BLOCK), 0, s, query, key, distance,
                           index, weight, eps, bpb, n1, n2, k);
    else
        hipLaunchKernelGGL((knn_register_kernel<T, KMAX, SOA, WEIGHTS>),
                           dim3((unsigned)(B * bpb)), dim3(KNN_BLOCK), 0, s, query, key, distance,
                           index, weight, eps, bpb, n1, n2, k);
}

// Whether knn_filter_launch takes this launch: the one test both entry points and the launch itself
// go by. Behind the wave kernel, which has the launches of few queries, it is the fastest route
// wherever a cloud holds 64 keys (timed against every other kernel here at 19000 to 262144 queries, 33 to
// 70000 keys, k = 3 to 32; us, others and this one: 19000 queries on 64 keys k = 3 12, 12, k = 16 22, 18,
// k = 32 28, 28; 65536 on 256, k = 8 33, 20, on 768, k = 16 97, 41, on 70000, k = 20 4470, 900; on 33
// keys k = 32 16, 20). A slot has 27 bits or more for its key, of 32 slots 26.
inline bool knn_filter_takes(int64_t B, int n1, int n2, int k)
{
    const int64_t bpb = ((int64_t)n1 + 255) / 256;
    return k <= 32 && n2 >= 64 && (k <= 4 || n2 <= (k <= 16 ? 1 << 27 : 1 << 26)) && B * bpb <= TK_MAX_I32;
}

template <int KMAX, bool SOA, bool WEIGHTS, int LANES, int KIND>
int knn_filter_launch_as(const float *query, const float *key, float *distance, int64_t *index,
                         float *weight, float eps, int64_t B, int n1, int n2, int k, hipStream_t s, bool halves = false)
{
    const int64_t bpb = ((int64_t)n1 + LANES - 1) / LANES;
    hipLaunchKernelGGL((knn_filter_kernel_f32<KMAX, SOA, WEIGHTS, LANES, KIND>), dim3((unsigned)(B * bpb), halves ? 2 : 1),
                       dim3(LANES), 0, s, query, key, distance, index, weight, eps, (int)bpb, n1, n2, k);
    return tk_launch_status();
}

template <int KMAX, bool SOA, bool WEIGHTS>
int knn_filter_launch(const float *query, const float *key, float *distance, int64_t *index,
                      float *weight, float eps, int64_t B, int n1, int n2, int k, hipStream_t s,
                      bool whatever_the_size = false)
{
    // 512 lanes: two workgroups (16 waves) per CU. A launch of few such workgroups leaves CUs without one: 256 lanes
    // then, unless there are keys enough for boxes. The times of the instances over that of the same kernel without
    // boxes and without keys put to all queries (256 lanes up to 128 or 160 workgroups of 512, else 512):
    //   8 x 4096 queries, in launches of few     every key, 256 lanes   512   boxes, unless ordered
    //     2048 keys in random order k = 3                 0.90           0.94          0.91
    //     2048 k = 8                                      0.89           0.99          0.96
    //     4096 k = 8                                      0.90           0.96          0.85
    //     4096 k = 16                                     0.94           1.08          1.01
    //     8192 k = 16                                     0.95           1.04          0.91
    //   16 x 8192, a workgroup to a CU: 4096 k = 16       1.02           0.96          0.91
    //     2048 k = 8                                      0.97           0.91          0.91 (in clusters 0.99, 0.92, 0.97)
    //   32 x 8192, two: 1024 k = 3                        1.04           0.87          0.87 (boxes; voxels in order 0.73)
    // Clouds of up to 256 queries have half of the 512 lanes to help with the staging, and one or two waves more to the
    // boxes' one: 200 x 120 on 4096 k = 8 1.07, 0.94; 80 x 250 on 8192 k = 16 0.95, 0.86, boxes 0.95; from 16384 keys
    // on boxes are even for k = 3, 0.89 and 0.83. 32 slots leave room for three waves per SIMD, twelve a CU: three
    // workgroups of 256 lanes or one of 512.
    if (!(whatever_the_size || knn_filter_takes(B, n1, n2, k)))
        return TK3D_ERR_UNSUPPORTED;
    const auto as = [&](auto lanes, auto kind, bool halves = false) {
        return knn_filter_launch_as<KMAX, SOA, WEIGHTS, decltype(lanes)::value, decltype(kind)::value>(
            query, key, distance, index, weight, eps, B, n1, n2, k, s, halves);
    };
    using Wide = std::integral_constant<int, 512>;
    using Narrow = std::integral_constant<int, 256>;
    using EveryKey = std::integral_constant<int, KNN_EVERY_KEY>;
    if constexpr (KMAX <= 16) {
        const int64_t wide = B * (((int64_t)n1 + 511) / 512), cus = tk_cu_count();
        const bool some = n1 > 256 || (n1 > 128 && n2 >= 4096 * KMAX);
        if (some && wide > cus && n2 >= 1024)
            return as(Wide{}, std::integral_constant<int, KNN_BOXES>{});
        const bool half = 2 * wide <= cus;
        if (some && wide <= cus && n2 >= (half ? 512 * KMAX : 128 * KMAX + 1536))
            return as(Wide{}, std::integral_constant<int, KNN_BOXES_UNLESS_ORDERED>{}, half);
        if (n1 <= 256 || wide > (KMAX <= 8 ? 128 : 160))
            return as(Wide{}, EveryKey{});
    }
    return as(Narrow{}, EveryKey{});
}

// Rows of k <= 64 results in place: ascending distance (equal ones in slot order, NaNs last, as a
// stable sort leaves them) if `sorted`, then square roots if `root`. W lanes to a row.
template <typename T, int W>
__global__ __launch_bounds__(KNN_BLOCK) void knn_rows_kernel(T *distance, int64_t *index, int64_t rows,
                                                             int k, int sorted, int root)
{
    const int lane = threadIdx.x & 63, at = lane & (W - 1), first = lane - at;
    const int64_t row = ((int64_t)blockIdx.x * KNN_BLOCK + threadIdx.x) / W;
    const bool mine = row < rows && at < k;
    T d = 0;
    int64_t i = 0;
    if (mine) {
        d = distance[row * k + at];
        i = index[row * k + at];
    }
    int place = at;
    if (sorted) {
        place = 0;
        for (int l = 0; l < k; ++l) {
            const T other = __shfl(d, first + l);
            const bool less = other < d || (d != d && other == other);
            const bool same = other == d || (d != d && other != other);
            place += less || (same && l < at) ? 1 : 0;
        }
    }
    if (root)
        d = sizeof(T) == 4 ? (T)__builtin_sqrtf((float)d) : (T)__builtin_sqrt((double)d);
    if (mine) {
        distance[row * k + place] = d;
        index[row * k + place] = i;
    }
}

template <typename T>
int knn_rows(T *distance, int64_t *index, int64_t rows, int k, int sorted, int root, hipStream_t s)
{
    const int width = k <= 8 ? 8 : k <= 16 ? 16 : k <= 32 ? 32 : 64;
    const int64_t blocks = (rows * width + KNN_BLOCK - 1) / KNN_BLOCK;
    if (k > 64 || blocks > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
#define TK_ROWS(W)                                                                             \
    hipLaunchKernelGGL((knn_rows_kernel<T, W>), dim3((unsigned)blocks), dim3(KNN_BLOCK), 0, s, \
                       distance, index, rows, k, sorted, root)
    if (width == 8)
        TK_ROWS(8);
    else if (width == 16)
        TK_ROWS(16);
    else if (width == 32)
        TK_ROWS(32);
    else
        TK_ROWS(64);
#undef TK_ROWS
    return tk_launch_status();
}

template <typename T>
int knn(const T *query, const T *key, int64_t B, int64_t N1, int64_t N2, int64_t k,
        int version, T *distance, int64_t *index, void *stream)
{
    if (B < 0 || N1 < 0 || N2 < 0)
        return TK3D_ERR_BAD_SIZE;
    if (version != 0 && version != 1)
        return TK3D_ERR_BAD_VERSION;
    if (k <= 0 || k > N2)
        return TK3D_ERR_BAD_K;
    if (N1 > TK_MAX_I32 / 4 || N2 > TK_MAX_I32 / 4 || !tk_fits(TK_MAX_ELEMS, B, N1, k) ||
        !tk_fits(TK_MAX_ELEMS, B, N2, 3))
        return TK3D_ERR_UNSUPPORTED;
    if (B * N1 == 0)
        return TK3D_OK;
    if (!query || !key || !distance || !index)
        return TK3D_ERR_NULL_POINTER;
    const int64_t bpb = (N1 + KNN_BLOCK - 1) / KNN_BLOCK;
    if (B * bpb > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    const int n1 = (int)N1, n2 = (int)N2, kk = (int)k;
    if constexpr (sizeof(T) == 4) {
        if (knn_wave_pays(B * N1, N2, kk))
            return knn_wave_launch<false, false>(query, key, distance, index, nullptr, 0.0f, B, n1,
                                                 n2, kk, 0, 0, s);
    }
    if (k <= 4) {
        // the pre-filtered kernel from 64 keys on, else the batched kernel
        if constexpr (sizeof(T) == 4) {
            const int rc = knn_filter_launch<4, false, false>(query, key, distance, index, nullptr,
                                                              0.0f, B, n1, n2, kk, s);
            if (rc != TK3D_ERR_UNSUPPORTED)
                return rc;
        }
        knn_launch<T, 4>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
    } else if constexpr (sizeof(T) == 4) {
        // fp32, k >= 5
        if (k <= 32) {
            // the pre-filtered kernel from 64 keys on
            const int rc =
                k <= 8 ? knn_filter_launch<8, false, false>(query, key, distance, index, nullptr,
                                                            0.0f, B, n1, n2, kk, s)
                : k <= 16
                    ? knn_filter_launch<16, false, false>(query, key, distance, index, nullptr,
                                                          0.0f, B, n1, n2, kk, s)
                    : knn_filter_launch<32, false, false>(query, key, distance, index, nullptr,
                                                          0.0f, B, n1, n2, kk, s);
            if (rc != TK3D_ERR_UNSUPPORTED)
                return rc;
        }
        // Slots in LDS as a tournament tree: more than 32 neighbours, and clouds of under 64 keys, on which launches
        // with k <= 8 below 131072 queries are a little faster with slots in registers.
        if (k <= 8 && B * N1 < 131072)
            knn_launch<T, 8>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 8)
            return knn_tree_launch<8>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 16)
            return knn_tree_launch<16>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 32)
            return knn_tree_launch<32>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 64)
            return knn_tree_launch<64>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 128)
            return knn_tree_launch<128>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 256 && n2 <= 65536)
            // 136 KiB of LDS per wave with 16-bit key indices: one wave per CU, still some
            // twenty times faster than keeping the slots in global memory
            return knn_tree_launch_as<256, true>(query, key, distance, index, B, n1, n2, kk, s);
        else
            hipLaunchKernelGGL((knn_global_kernel<T>), dim3((unsigned)(B * bpb)),
                               dim3(KNN_BLOCK), 0, s, query, key, distance, index, (int)bpb,
                               n1, n2, kk);
    } else {
        // fp64: slots in registers up to k = 16, the LDS tree beyond (k = 64 at B=32,
        // 2048 x 8192: the register variant pays 2 k selects per insertion on 64-bit values)
        if (k <= 8)
            knn_launch<T, 8>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 16)
            knn_launch<T, 16>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 32)
            return knn_tree_launch<32, T>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 64)
            return knn_tree_launch<64, T>(query, key, distance, index, B, n1, n2, kk, s);
        else if (k <= 128)
            return knn_tree_launch<128, T>(query, key, distance, index, B, n1, n2, kk, s);
        else
            hipLaunchKernelGGL((knn_global_kernel<T>), dim3((unsigned)(B * bpb)),
                               dim3(KNN_BLOCK), 0, s, query, key, distance, index, (int)bpb,
                               n1, n2, kk);
    }
    return tk_launch_status();
}

// KNN on [B,3,N] clouds with the kernels that read either layout, k <= 64 (beyond:
// TK3D_ERR_UNSUPPORTED before anything is launched; the caller copies the clouds and calls
// knn()). fp32: the wave and pre-filtered kernels where knn() would launch them, else the batched kernel
// for k <= 4 and the LDS tree kernel. fp64: slots in registers.
template <typename T>
int knn_bcn(const T *query, const T *key, int64_t B, int64_t N1, int64_t N2, int64_t k,
            int version, T *distance, int64_t *index, void *stream)
{
    if (B < 0 || N1 < 0 || N2 < 0)
        return TK3D_ERR_BAD_SIZE;
    if (version != 0 && version != 1)
        return TK3D_ERR_BAD_VERSION;
    if (k <= 0 || k > N2)
        return TK3D_ERR_BAD_K;
    if (N1 > TK_MAX_I32 / 4 || N2 > TK_MAX_I32 / 4 || !tk_fits(TK_MAX_ELEMS, B, N1, k) ||
        !tk_fits(TK_MAX_ELEMS, B, N2, 3) || k > 64)
        return TK3D_ERR_UNSUPPORTED;
    const int64_t bpb = (N1 + KNN_BLOCK - 1) / KNN_BLOCK;
    if (B * bpb > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
    const int n1 = (int)N1, n2 = (int)N2, kk = (int)k;
    if (B * N1 == 0)
        return TK3D_OK;
    if (!query || !key || !distance || !index)
        return TK3D_ERR_NULL_POINTER;
    hipStream_t s = (hipStream_t)stream;
    if constexpr (sizeof(T) == 4) {
        if (knn_wave_pays(B * N1, N2, kk))
            return knn_wave_launch<true, false>(query, key, distance, index, nullptr, 0.0f, B, n1, n2,
                                                kk, 0, 0, s);
        if (k > 4 && !knn_filter_takes(B, n1, n2, kk)) {
            // more than 32 neighbours, or fewer than 64 keys: the LDS tree, reading the coordinate planes
            if (k <= 8)
                return knn_tree_launch<8, float, true>(query, key, distance, index, B, n1, n2, kk, s);
            if (k <= 16)
                return knn_tree_launch<16, float, true>(query, key, distance, index, B, n1, n2, kk, s);
            if (k <= 32)
                return knn_tree_launch<32, float, true>(query, key, distance, index, B, n1, n2, kk, s);
            return knn_tree_launch<64, float, true>(query, key, distance, index, B, n1, n2, kk, s);
        }
        int rc = TK3D_ERR_UNSUPPORTED;
        if (k <= 4) {
            rc = knn_filter_launch<4, true, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                   n1, n2, kk, s);
            if (rc == TK3D_ERR_UNSUPPORTED) {
                knn_launch<T, 4, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
                rc = tk_launch_status();
            }
        } else if (k <= 8) {
            rc = knn_filter_launch<8, true, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                   n1, n2, kk, s);
        } else if (k <= 16) {
            rc = knn_filter_launch<16, true, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                    n1, n2, kk, s);
        } else {
            rc = knn_filter_launch<32, true, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                    n1, n2, kk, s);
        }
        return rc;
    } else {
        if (k <= 4)
            knn_launch<T, 4, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 8)
            knn_launch<T, 8, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 16)
            knn_launch<T, 16, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else if (k <= 32)
            knn_launch<T, 32, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        else
            knn_launch<T, 64, true>(query, key, distance, index, B, (int)bpb, n1, n2, kk, s);
        return tk_launch_status();
    }
}

// KNN with the rows put in order and the square roots taken on the way out, k <= 64.
template <typename T>
int knn_ordered(const T *query, const T *key, bool channels_first, int64_t B, int64_t N1, int64_t N2,
                int64_t k, int sorted, int root, T *distance, int64_t *index, void *stream)
{
    if (k > 64)
        return TK3D_ERR_UNSUPPORTED;
    if constexpr (sizeof(T) == 4) {
        if (B > 0 && N1 > 0 && k > 0 && k <= N2 && query && key && distance && index &&
            N1 <= TK_MAX_I32 / 4 && N2 <= TK_MAX_I32 / 4 && tk_fits(TK_MAX_ELEMS, B, N2, 3) &&
            knn_wave_pays(B * N1, N2, (int)k)) {
            const auto launch = channels_first ? knn_wave_launch<true, false> : knn_wave_launch<false, false>;
            return launch(query, key, distance, index, nullptr, 0.0f, B, (int)N1, (int)N2, (int)k,
                          sorted, root, (hipStream_t)stream);
        }
    }
    const int rc = channels_first ? knn_bcn<T>(query, key, B, N1, N2, k, 1, distance, index, stream)
                                  : knn<T>(query, key, B, N1, N2, k, 1, distance, index, stream);
    if (rc != TK3D_OK || B * N1 == 0 || !(sorted || root))
        return rc;
    return knn_rows<T>(distance, index, B * N1, (int)k, sorted, root, (hipStream_t)stream);
}

// 3 nearest neighbours with the interpolation weights formed in the same kernel.
template <typename T>
int three_nn(const T *query, const T *key, bool channels_first, int64_t B, int64_t N1,
             int64_t N2, double eps, T *distance, int64_t *index, T *weight, void *stream)
{
    if (B < 0 || N1 < 0 || N2 < 0)
        return TK3D_ERR_BAD_SIZE;
    if (N2 < 3)
        return TK3D_ERR_BAD_K;
    if (N1 > TK_MAX_I32 / 4 || N2 > TK_MAX_I32 / 4 || !tk_fits(TK_MAX_ELEMS, B, N1, 3) ||
        !tk_fits(TK_MAX_ELEMS, B, N2, 3))
        return TK3D_ERR_UNSUPPORTED;
    if (B * N1 == 0)
        return TK3D_OK;
    if (!query || !key || !distance || !index || !weight)
        return TK3D_ERR_NULL_POINTER;
    const int64_t bpb = (N1 + KNN_BLOCK - 1) / KNN_BLOCK;
    if (B * bpb > TK_MAX_I32)
        return TK3D_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    if constexpr (sizeof(T) == 4) {
        if (knn_wave_pays(B * N1, N2, 3)) {
            const auto launch = channels_first ? knn_wave_launch<true, true> : knn_wave_launch<false, true>;
            return launch(query, key, distance, index, weight, (float)eps, B, (int)N1, (int)N2, 3, 0, 0,
                          s);
        }
        const int rf = channels_first
                           ? knn_filter_launch<4, true, true>(query, key, distance, index, weight,
                                                              (float)eps, B, (int)N1, (int)N2, 3, s)
                           : knn_filter_launch<4, false, true>(query, key, distance, index, weight,
                                                               (float)eps, B, (int)N1, (int)N2, 3,
                                                               s);
        if (rf != TK3D_ERR_UNSUPPORTED)
            return rf;
    }
    if (channels_first)
        knn_launch<T, 4, true, true>(query, key, distance, index, B, (int)bpb, (int)N1, (int)N2,
                                     3, s, weight, (T)eps);
    else
        knn_launch<T, 4, false, true>(query, key, distance, index, B, (int)bpb, (int)N1,
                                      (int)N2, 3, s, weight, (T)eps);
    return tk_launch_status();
}

}  // namespace

extern "C" {

int tk3d_three_nn_f32(const float *query, const float *key, int channels_first, int64_t B,
                      int64_t N1, int64_t N2, double eps, float *distance, int64_t *index,
                      float *weight, void *stream)
{
    return three_nn<float>(query, key, channels_first != 0, B, N1, N2, eps, distance, index,
                           weight, stream);
}

int tk3d_three_nn_f64(const double *query, const double *key, int channels_first, int64_t B,
                      int64_t N1, int64_t N2, double eps, double *distance, int64_t *index,
                      double *weight, void *stream)
{
    return three_nn<double>(query, key, channels_first != 0, B, N1, N2, eps, distance, index,
                            weight, stream);
}

int tk3d_knn_distance_bcn_f32(const float *query, const float *key, int64_t B, int64_t N1,
                              int64_t N2, int64_t k, int version, float *distance,
                              int64_t *index, void *stream)
{
    return knn_bcn<float>(query, key, B, N1, N2, k, version, distance, index, stream);
}

int tk3d_knn_distance_bcn_f64(const double *query, const double *key, int64_t B, int64_t N1,
                              int64_t N2, int64_t k, int version, double *distance,
                              int64_t *index, void *stream)
{
    return knn_bcn<double>(query, key, B, N1, N2, k, version, distance, index, stream);
}

int tk3d_knn_distance_f32(const float *query, const float *key, int64_t B, int64_t N1,
                          int64_t N2, int64_t k, int version, float *distance,
                          int64_t *index, void *stream)
{
    return knn<float>(query, key, B, N1, N2, k, version, distance, index, stream);
}

int tk3d_knn_distance_f64(const double *query, const double *key, int64_t B, int64_t N1,
                          int64_t N2, int64_t k, int version, double *distance,
                          int64_t *index, void *stream)
{
    return knn<double>(query, key, B, N1, N2, k, version, distance, index, stream);
}

int tk3d_knn_distance_ordered_f32(const float *query, const float *key, int channels_first,
                                  int64_t B, int64_t N1, int64_t N2, int64_t k, int sorted, int root,
                                  float *distance, int64_t *index, void *stream)
{
    return knn_ordered<float>(query, key, channels_first != 0, B, N1, N2, k, sorted, root, distance,
                              index, stream);
}

int tk3d_knn_distance_ordered_f64(const double *query, const double *key, int channels_first,
                                  int64_t B, int64_t N1, int64_t N2, int64_t k, int sorted, int root,
                                  double *distance, int64_t *index, void *stream)
{
    return knn_ordered<double>(query, key, channels_first != 0, B, N1, N2, k, sorted, root, distance,
                               index, stream);
}

int64_t tk3d_debug_knn_wave_queries(int64_t keys, int64_t k) { return knn_wave_queries(keys, k); }

int tk3d_debug_knn_wave_f32(const float *query, const float *key, int channels_first, int64_t B,
                            int64_t N1, int64_t N2, int64_t k, float *distance, int64_t *index,
                            void *stream)
{
    if (B < 0 || N1 < 0 || N2 < 0)
        return TK3D_ERR_BAD_SIZE;
    if (k <= 0 || k > N2)
        return TK3D_ERR_BAD_K;
    if (N1 > TK_MAX_I32 / 4 || N2 > TK_MAX_I32 / 4 || !tk_fits(TK_MAX_ELEMS, B, N1, k) ||
        !tk_fits(TK_MAX_ELEMS, B, N2, 3))
        return TK3D_ERR_UNSUPPORTED;
    if (B * N1 == 0)
        return TK3D_OK;
    if (!query || !key || !distance || !index)
        return TK3D_ERR_NULL_POINTER;
    hipStream_t s = (hipStream_t)stream;
    const auto launch = channels_first ? knn_wave_launch<true, false> : knn_wave_launch<false, false>;
    return launch(query, key, distance, index, nullptr, 0.0f, B, (int)N1, (int)N2, (int)k, 0, 0, s);
}

int tk3d_debug_knn_filter_f32(const float *query, const float *key, int64_t B, int64_t N1,
                              int64_t N2, int64_t k, float *distance, int64_t *index,
                              void *stream)
{
    if (B < 0 || N1 < 0 || N2 < 0)
        return TK3D_ERR_BAD_SIZE;
    if (k <= 0 || k > N2)
        return TK3D_ERR_BAD_K;
    if (k > 32 || N1 > TK_MAX_I32 / 4 || N2 > TK_MAX_I32 / 4 ||
        !tk_fits(TK_MAX_ELEMS, B, N1, k) || !tk_fits(TK_MAX_ELEMS, B, N2, 3) ||
        N2 > ((int64_t)1 << 26) || !tk_fits(TK_MAX_I32, B, (N1 + 255) / 256))
        return TK3D_ERR_UNSUPPORTED;
    if (B * N1 == 0)
        return TK3D_OK;
    if (!query || !key || !distance || !index)
        return TK3D_ERR_NULL_POINTER;
    hipStream_t s = (hipStream_t)stream;
    const int n1 = (int)N1, n2 = (int)N2, kk = (int)k;
    if (k <= 4)
        return knn_filter_launch<4, false, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                  n1, n2, kk, s, true);
    if (k <= 8)
        return knn_filter_launch<8, false, false>(query, key, distance, index, nullptr, 0.0f, B,
                                                  n1, n2, kk, s, true);
    if (k <= 16)
        return knn_filter_launch<16, false, false>(query, key, distance, index, nullptr, 0.0f, B, n1,
                                                   n2, kk, s, true);
    return knn_filter_launch<32, false, false>(query, key, distance, index, nullptr, 0.0f, B, n1, n2,
                                               kk, s, true);
}

}  // extern "C"
