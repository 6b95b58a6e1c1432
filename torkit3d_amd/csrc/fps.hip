// Farthest point sampling for gfx950.
//
// Clouds that fit in one workgroup's registers (16384 points in fp32, 8192 in fp64) are
// sampled by one workgroup each; larger ones by one launch of many workgroups per
// selection step (fps_wide_step_kernel, further down). The K-1 selection steps are
// strictly serial, so the one-workgroup kernels are built for latency per step, not
// throughput:
//   * every lane keeps P points and their running minimum distance in registers
//     for the whole kernel - the loop touches no global memory except the one
//     index it emits per step;
//   * per step a lane updates its P minima and finds its local maximum, the wave
//     reduces with DPP row shifts / row broadcasts (no LDS), ballot + find-first
//     pick the winning lane on the scalar unit;
//   * waves exchange (value, point index, xyz) through double-buffered LDS slots,
//     so a step costs a single s_barrier, and every wave redoes the tiny
//     cross-wave reduction itself instead of waiting for a broadcast.
//
// Ties. The reference resolves equal maxima by its thread layout: thread t scans
// j = t, t+BS, ... keeping the first maximum, then a shared-memory tree keeps the
// left operand (sample_farthest_points_kernel.cu:46-72, :75-95), i.e. the winner
// is the candidate with the smallest (bit-reversed t, j / BS). The points are
// laid out here in exactly that priority order ("positions"), lanes take
// consecutive positions, and every reduction keeps the lowest position among
// equal values, which reproduces the reference's choice.
#include <type_traits>

#include "tk3d_common.h"
#include "tk3d_curve.h"

namespace {

template <typename T> struct Bits;
template <> struct Bits<float> { using type = int; };
template <> struct Bits<double> { using type = long long; };

template <int CTRL, int ROW_MASK> __device__ __forceinline__ float dpp_move(float v)
{
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v),
                                           __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF,
                                           false));
}
template <int CTRL, int ROW_MASK> __device__ __forceinline__ double dpp_move(double v)
{
    const long long b = __builtin_bit_cast(long long, v);
    int lo = (int)b, hi = (int)(b >> 32);
    lo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xF, false);
    hi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xF, false);
    return __builtin_bit_cast(double,
                              ((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ float read_lane(float v, int lane)
{
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ int read_lane(int v, int lane)
{
    return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ double read_lane(double v, int lane)
{
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}

// Maximum over the 64 lanes, returned as a wave-uniform value. Inclusive scan
// inside each row of 16 (row_shr 1,2,4,8), then row_bcast15 / row_bcast31 carry
// the row totals up so that lane 63 holds the result.
template <typename T> __device__ __forceinline__ T wave_max(T v)
{
    if constexpr (std::is_same<T, float>::value)
        return tk_wave_extreme<true>(v);
    v = tk_max<T>(v, dpp_move<0x111, 0xF>(v));
    v = tk_max<T>(v, dpp_move<0x112, 0xF>(v));
    v = tk_max<T>(v, dpp_move<0x114, 0xF>(v));
    v = tk_max<T>(v, dpp_move<0x118, 0xF>(v));
    v = tk_max<T>(v, dpp_move<0x142, 0xA>(v));
    v = tk_max<T>(v, dpp_move<0x143, 0xC>(v));
    return read_lane(v, 63);
}

// Coordinate `a` of point `j`: clouds are [n,3] rows, or with SOA three planes [3,n]
// (the layout the reference's models keep their clouds in).
template <bool SOA, typename T>
__device__ __forceinline__ T fps_coord(const T *__restrict__ pts, int n, int64_t j, int a)
{
    return SOA ? pts[(int64_t)a * n + j] : pts[j * 3 + a];
}

struct FpsLayout {
    int n;        // points per cloud
    int k;        // samples per cloud
    int bs;       // the reference's block size for this n (power of two, 32..512)
    int log2_bs;
    int c;        // ceil(n / bs): points per reference thread
    float inv_c;  // 1 / c
};

// Point index of a position in the priority order described at the top.
__device__ __forceinline__ int fps_point_of_position(int pos, const FpsLayout &L)
{
    int r = (int)(((float)pos + 0.5f) * L.inv_c);
    // One correction step makes the float estimate exact for every pos < 2^24.
    r += ((r + 1) * L.c <= pos) ? 1 : 0;
    r -= (r * L.c > pos) ? 1 : 0;
    const int cc = pos - r * L.c;
    const int t = (int)(__builtin_bitreverse32((unsigned)r) >> (32 - L.log2_bs));
    return t + cc * L.bs;
}

// One selection step per exchange between the waves, on points and minima held in
// registers (lane `tid` holds positions tid * P .. tid * P + P - 1). fmin keeps a
// minimum when a later distance is NaN, as the reference's '>' does. `md` arrives
// holding the distances to point 0 (see fps_first_minimum).
template <typename T, int P, int NT>
__device__ __forceinline__ void fps_one_step_loop(int64_t *__restrict__ out, const FpsLayout &L,
                                                  const T (&x)[P], const T (&y)[P],
                                                  const T (&z)[P], T (&md)[P], T cx, T cy, T cz)
{
    constexpr int NW = NT / TK_WAVE;
    __shared__ T s_val[2][NW], s_x[2][NW], s_y[2][NW], s_z[2][NW];
    __shared__ int s_j[2][NW];
    const int tid = threadIdx.x;
    const int lane = tid & (TK_WAVE - 1);
    const int wave = tid / TK_WAVE;
    int sel_j = 0;
    if (tid == 0)
        out[0] = 0;

    for (int it = 1; it < L.k; ++it) {
        // Lane-local update and first maximum above zero (strict '>' from zero, as
        // the reference thread does).
        T best = (T)0;
        int bp = 0;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const T d = tk_dist2<T>(x[p], y[p], z[p], cx, cy, cz);
            md[p] = tk_min<T>(md[p], d);
            const bool up = md[p] > best;
            best = up ? md[p] : best;
            bp = up ? p : bp;
        }
        const T wmax = wave_max<T>(best);
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(best == wmax);
        const int wl = __builtin_ctzll(hit);  // lowest lane holding the maximum
        const int wp = read_lane(bp, wl);
        T sx = x[0], sy = y[0], sz = z[0];
#pragma unroll
        for (int p = 1; p < P; ++p) {
            if (wp == p) {  // wave-uniform: a scalar branch
                sx = x[p];
                sy = y[p];
                sz = z[p];
            }
        }
        // Cross-lane reads happen with the whole wave active: a lane switched off
        // by a branch has no defined value to hand over.
        const T wx = read_lane(sx, wl), wy = read_lane(sy, wl), wz = read_lane(sz, wl);
        const int wj = fps_point_of_position((wave * TK_WAVE + wl) * P + wp, L);
        const int buf = it & 1;
        if (lane == 0) {
            s_val[buf][wave] = wmax;
            s_j[buf][wave] = wj;
            s_x[buf][wave] = wx;
            s_y[buf][wave] = wy;
            s_z[buf][wave] = wz;
        }
        __syncthreads();
        // Every wave reduces the NW candidates itself. Lower waves hold lower
        // positions, so the lowest lane among equal values is the right winner.
        const bool has = lane < NW;
        const T cv = has ? s_val[buf][has ? lane : 0] : (T)-1;
        const T gmax = wave_max<T>(cv);
        if (gmax > (T)0) {
            const int gl = __builtin_ctzll(__builtin_amdgcn_ballot_w64(cv == gmax));
            sel_j = s_j[buf][gl];
            cx = s_x[buf][gl];
            cy = s_y[buf][gl];
            cz = s_z[buf][gl];
        }
        // gmax == 0: no point lies away from the chosen set; the previous choice
        // is emitted again, as the reference does.
        if (tid == 0)
            out[it] = (int64_t)sel_j;
    }
}

// The reference's minima start "unset" and take whatever the first step computes
// (sample_farthest_points_kernel.cu:59-64), a NaN included, which then never compares
// above anything. So a minimum starts at the distance to point 0, with -1 for a NaN and
// for unused slots: min() keeps -1 and it never exceeds 0.
template <typename T> __device__ __forceinline__ T fps_first_minimum(bool used, T d0)
{
    return (used && d0 == d0) ? d0 : (T)-1;
}

// The whole sampling of one cloud with the plain loop.
template <typename T, int P, int NT, bool SOA>
__device__ __forceinline__ void fps_plain(const T *__restrict__ pts, int64_t *__restrict__ out,
                                          const FpsLayout &L)
{
    const int tid = threadIdx.x;
    T x[P], y[P], z[P], md[P];
    const int npos = L.bs * L.c;
    const T cx = fps_coord<SOA>(pts, L.n, 0, 0), cy = fps_coord<SOA>(pts, L.n, 0, 1),
            cz = fps_coord<SOA>(pts, L.n, 0, 2);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pos = tid * P + p;
        const int j = pos < npos ? fps_point_of_position(pos, L) : L.n;
        const bool ok = j < L.n;
        x[p] = ok ? fps_coord<SOA>(pts, L.n, j, 0) : (T)0;
        y[p] = ok ? fps_coord<SOA>(pts, L.n, j, 1) : (T)0;
        z[p] = ok ? fps_coord<SOA>(pts, L.n, j, 2) : (T)0;
        md[p] = fps_first_minimum<T>(ok, tk_dist2<T>(x[p], y[p], z[p], cx, cy, cz));
    }
    fps_one_step_loop<T, P, NT>(out, L, x, y, z, md, cx, cy, cz);
}

// fps_plain as a kernel. With `only_odd` it does so only for a cloud that holds a NaN or an
// infinite coordinate, and returns at once for any other.
//
// The fp32 kernel below assumes finite coordinates (minima ordered as integers, a selected
// point's minimum dropping to zero) and is followed by this one with `only_odd`, which
// redoes the rare cloud it got wrong the way the reference treats it: a NaN point is never
// selected, an infinite one, once selected, is selected at every later step. The check
// lives here rather than in that kernel because anything added to it, even a test in
// its prologue, moved its loop's code and cost 4-7 % at 32 points per lane; the extra
// launch costs a few microseconds.
template <typename T, int P, int NT, bool SOA>
__global__ __launch_bounds__(NT) void fps_register_kernel(const T *__restrict__ points,
                                                          int64_t *__restrict__ index,
                                                          FpsLayout L, int only_odd)
{
    const T *__restrict__ pts = points + (int64_t)blockIdx.x * L.n * 3;
    int64_t *__restrict__ out = index + (int64_t)blockIdx.x * L.k;
    const int tid = threadIdx.x;
    if (only_odd) {
        // v - v is zero exactly for finite v; the 3n values are scanned in memory order
        bool odd = false;
#pragma unroll 8
        for (int i = tid; i < L.n * 3; i += NT) {
            const T v = pts[i];
            odd |= !(v - v == (T)0);
        }
        if (!__syncthreads_or(odd ? 1 : 0))  // uniform over the workgroup
            return;
    }
    fps_plain<T, P, NT, SOA>(pts, out, L);
}

// ---- fp32 fast path ------------------------------------------------------------
// Same algorithm as fps_register_kernel, tuned for the serial step:
//   * running minima are kept as the bit patterns of non-negative floats, which
//     order like signed integers; integer min/max need no NaN canonicalisation
//     and the -1.0f marker of unused slots (a negative integer) stays put;
//   * a lane reduces its P minima through a binary tree of maxima kept in
//     registers; the wave's maximum is a scan with DPP row shifts and broadcasts, and
//     the runner-up (the largest value of the other lanes) a second such scan that runs
//     beside the walk below;
//   * the winning lane comes from one ballot + scalar find-first; its winning
//     point is found by walking the winner lane's tree with v_readlane and
//     scalar branches (left child first = lowest position), and the leaf reached
//     reads that point's coordinates from fixed registers - log2(P) steps, no
//     per-point compares or select chains in the loop;
//   * a wave publishes its candidate (xyz, value) and (runner-up, point) in LDS; after the
//     single barrier every wave loads all candidates and decides by itself how many of
//     them are winners (see fps_multistep_kernel_f32).

struct FpsPick {
    float x, y, z;
    int j;
};

// Largest of the 64 lanes' values (all >= 0), wave-uniform: a scan along rows of 16 lanes
// with row shifts, the rows' results carried on with row broadcasts, the total read from
// lane 63. A lane without a source lane in a step takes 0.
__device__ __forceinline__ int wave_max_i32(int v)
{
#define TK3D_MAX_STEP(ctrl, rows)                                                      \
    {                                                                                  \
        const int o = __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, false);       \
        v = o > v ? o : v;                                                             \
    }
    TK3D_MAX_STEP(0x111, 0xf)  // row_shr:1
    TK3D_MAX_STEP(0x112, 0xf)  // row_shr:2
    TK3D_MAX_STEP(0x114, 0xf)  // row_shr:4
    TK3D_MAX_STEP(0x118, 0xf)  // row_shr:8
    TK3D_MAX_STEP(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
    TK3D_MAX_STEP(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef TK3D_MAX_STEP
    return __builtin_amdgcn_readlane(v, 63);
}

// The walk through a lane's tree of maxima from the root to the first leaf equal to `wmax`, which also reports the
// largest value it passed by: it sees the sibling of every node on its path, and the
// largest of those siblings is the lane's second-largest minimum (equal to `wmax` when
// the lane holds the maximum twice).
template <int P, int NODE> struct FpsWalk2 {
    static __device__ __forceinline__ void go(const int (&t)[2 * P], const float (&x)[P],
                                              const float (&y)[P], const float (&z)[P],
                                              const int (&jv)[P], int wl, int wmax,
                                              FpsPick &out, int &passed)
    {
        if constexpr (NODE >= P) {
            constexpr int p = NODE - P;
            out.x = read_lane(x[p], wl);
            out.y = read_lane(y[p], wl);
            out.z = read_lane(z[p], wl);
            out.j = read_lane(jv[p], wl);
            asm volatile("" ::"s"(out.j));
        } else {
            const int left = read_lane(t[2 * NODE], wl);
            const int right = read_lane(t[2 * NODE + 1], wl);
            if (left == wmax) {
                passed = right > passed ? right : passed;
                FpsWalk2<P, 2 * NODE>::go(t, x, y, z, jv, wl, wmax, out, passed);
            } else {
                passed = left > passed ? left : passed;
                FpsWalk2<P, 2 * NODE + 1>::go(t, x, y, z, jv, wl, wmax, out, passed);
            }
        }
    }
};

// fp32 kernel that takes up to MAXM selection steps per cross-wave exchange.
//
// A step's fixed cost (wave reduction, slot exchange, barrier: about 1000 clocks) is
// several times the cost of updating the minima for one more centre, so after the
// exchange every wave checks, redundantly, whether the next winners are already known.
// Let the waves' candidates be sorted by (value descending, wave ascending) - waves
// hold ascending position ranges, so this is the reference's order - and let w1 be the
// winner. The m-th candidate w_m (value V_m > 0) is the winner of the m-th following
// step exactly when
//   * no wave that already supplied a winner holds another point at or above V_m (each
//     wave publishes its second-largest minimum for this; ties are refused), and
//   * the canonical distance from w_m to every winner accepted so far is >= V_m, so the
//     coming updates leave its minimum at V_m;
// every other point is at or below V_m by the sort, minima only shrink, and the
// accepted winners drop to zero. The chain stops at the first candidate that fails;
// on uniform clouds about 2.7 steps are taken per exchange.
//
// The check is a chain of dependent instructions issued by one wave, so its length in
// instructions is its cost: conditions are single compares whose lane masks are combined
// in scalar registers, and the accepted candidates never go back to LDS - the coming
// update reads their coordinates with v_readlane from the lanes that already hold them.
template <int P, int NT, bool SOA, int MAXM>
__global__ __launch_bounds__(NT) void fps_multistep_kernel_f32(const float *__restrict__ points,
                                                               int64_t *__restrict__ index,
                                                               FpsLayout L)
{
    static_assert((P & (P - 1)) == 0, "P must be a power of two");
    constexpr int NW = NT / TK_WAVE;
    static_assert(NW <= 8, "the cross-wave step relates 8 x 8 candidates");
    constexpr int F32_INF = 0x7f800000;
    constexpr int F32_NEG1 = (int)0xbf800000;
    __shared__ float4 s_cand[2][8];  // a wave's candidate: x, y, z, running minimum (bits)
    __shared__ int2 s_aux[2][8];     // the wave's second-largest minimum, the candidate's index

    const int tid = threadIdx.x;
    const int lane = tid & (TK_WAVE - 1);
    const int wave = tid / TK_WAVE;
    const float *__restrict__ pts = points + (int64_t)blockIdx.x * L.n * 3;
    int64_t *__restrict__ out = index + (int64_t)blockIdx.x * L.k;

    float x[P], y[P], z[P];
    int jv[P];
    int t[2 * P];  // t[P + p]: running minimum of point p (bits); t[1..P-1]: maxima
    const int npos = L.bs * L.c;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pos = tid * P + p;
        const int j = pos < npos ? fps_point_of_position(pos, L) : L.n;
        const bool ok = j < L.n;
        x[p] = ok ? fps_coord<SOA>(pts, L.n, j, 0) : 0.0f;
        y[p] = ok ? fps_coord<SOA>(pts, L.n, j, 1) : 0.0f;
        z[p] = ok ? fps_coord<SOA>(pts, L.n, j, 2) : 0.0f;
        jv[p] = j;
        t[P + p] = ok ? F32_INF : F32_NEG1;
    }
    t[0] = 0;

    // Lane (a, b) = (lane / 8, lane % 8) relates candidate a to candidate b after an
    // exchange. The centres of the coming update are the candidates of the lanes in
    // `centres` (lane 8 a stands for candidate a); the first update is point 0.
    const int ca = lane >> 3, cb = lane & 7;
    float ax = fps_coord<SOA>(pts, L.n, 0, 0);
    float ay = fps_coord<SOA>(pts, L.n, 0, 1);
    float az = fps_coord<SOA>(pts, L.n, 0, 2);
    unsigned long long centres = 1ull;
    // the last point emitted is the candidate of lane ctz(last_mask) / 8, whose index that
    // lane keeps in last_j; no mask: point 0
    unsigned long long last_mask = 0ull;
    int last_j = 0;
    constexpr unsigned long long FIRST_OF_EIGHT = 0x0101010101010101ull;  // lanes b == 0
    constexpr unsigned long long EARLIER = 0x7f3f1f0f07030100ull;         // lanes b < a
    int nc = 1;
    if (tid == 0)
        out[0] = 0;
    if (tid < 16 && (tid & 7) >= NW) {  // waves that do not exist never have a candidate
        s_cand[tid >> 3][tid & 7] = make_float4(0.0f, 0.0f, 0.0f, -1.0f);
        s_aux[tid >> 3][tid & 7] = make_int2(0, 0);
    }

    int round = 0;
    for (int it = 1; it < L.k; it += nc, ++round) {
        for (unsigned long long todo = centres; todo != 0ull; todo &= todo - 1) {  // uniform
            const int l = __builtin_ctzll(todo);
            const float sx = read_lane(ax, l), sy = read_lane(ay, l), sz = read_lane(az, l);
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const float d = tk_dist2<float>(x[p], y[p], z[p], sx, sy, sz);
                const int db = __builtin_bit_cast(int, d);
                t[P + p] = t[P + p] < db ? t[P + p] : db;
            }
        }
#pragma unroll
        for (int i = P - 1; i >= 1; --i)
            t[i] = t[2 * i] > t[2 * i + 1] ? t[2 * i] : t[2 * i + 1];
        // Only points strictly above zero are candidates (the reference starts its
        // scan from max_dist = 0 with strict '>').
        const int best = t[1] > 0 ? t[1] : 0;
        const int wmax = wave_max_i32(best);
        const int wl = __builtin_ctzll(__builtin_amdgcn_ballot_w64(best == wmax));
        int second = wave_max_i32(lane == wl ? 0 : best);  // over the other lanes
        FpsPick pick;
        FpsWalk2<P, 1>::go(t, x, y, z, jv, wl, wmax, pick, second);  // and inside lane wl
        const int buf = round & 1;
        if (lane == 0) {
            s_cand[buf][wave] = make_float4(pick.x, pick.y, pick.z, __builtin_bit_cast(float, wmax));
            s_aux[buf][wave] = make_int2(second, pick.j);
        }
        __syncthreads();
        // Every wave now works out, redundantly and without a serial chain, how many of
        // the candidates are certain winners of the coming steps. All 64 lanes are active,
        // so conditions are combined as lane masks in scalar registers.
        const float4 A = s_cand[buf][ca], Bc = s_cand[buf][cb];
        const int2 Bx = s_aux[buf][cb];  // the wave's second-largest minimum, its point
        ax = A.x;
        ay = A.y;
        az = A.z;
        const int va = __builtin_bit_cast(int, A.w), vb = __builtin_bit_cast(int, Bc.w);
        // b comes before a in the reference's order: larger value, then lower position
        // (waves hold ascending ranges of positions)
        const unsigned long long m_before =
            __builtin_amdgcn_ballot_w64(vb > va) | (__builtin_amdgcn_ballot_w64(vb == va) & EARLIER);
        const unsigned long long m_live = __builtin_amdgcn_ballot_w64(va > 0);
        const float dab = tk_dist2<float>(A.x, A.y, A.z, Bc.x, Bc.y, Bc.z);
        // a survives b's selection: b's update leaves a's minimum alone, and b's wave
        // holds nothing else at or above it
        const unsigned long long m_far =
            __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int, dab) >= va);
        const unsigned long long m_alone = __builtin_amdgcn_ballot_w64(Bx.x < va);
        const unsigned long long m_fine = ~m_before | (m_far & m_alone);
        // byte a of a mask: candidate a against every b
        const unsigned before_a =
            __builtin_amdgcn_ubfe(lane < 32 ? (unsigned)m_before : (unsigned)(m_before >> 32),
                                  (unsigned)(lane & 24), 8u);
        const unsigned fine_a =
            __builtin_amdgcn_ubfe(lane < 32 ? (unsigned)m_fine : (unsigned)(m_fine >> 32),
                                  (unsigned)(lane & 24), 8u);
        const int rank = __builtin_popcount(before_a);  // a permutation of the candidates
        const unsigned long long fine = __builtin_amdgcn_ballot_w64(fine_a == 0xffu) & m_live;
        // Lane (a, b) asks whether candidate a has rank b and passed; folding the bytes of
        // that mask together gives, in bit b, whether the candidate of rank b passed.
        unsigned long long passed = __builtin_amdgcn_ballot_w64(rank == cb) & fine;
        passed |= passed >> 32;
        passed |= passed >> 16;
        passed |= passed >> 8;
        const int left = L.k - it;  // steps still wanted
        int good = __builtin_ctz(~(unsigned)passed | (1u << MAXM));  // ranks 0..good-1 passed
        good = good < left ? good : left;
        centres = __builtin_amdgcn_ballot_w64(rank < good) & FIRST_OF_EIGHT;
        if (good > 0) {  // uniform
            if (wave == 0) {  // uniform
                if (ca == cb && rank < good)
                    out[it + rank] = (int64_t)Bx.y;
            }
            // the last point emitted, should the cloud run out of distinct points
            last_mask = __builtin_amdgcn_ballot_w64(rank == good - 1);
            last_j = Bx.y;
            nc = good;
        } else {
            // No point lies away from the chosen set: the previous choice is emitted again,
            // as the reference does. Every minimum is zero already: nothing is updated.
            if (tid == 0)
                out[it] = last_mask != 0ull
                              ? (int64_t)read_lane(last_j, __builtin_ctzll(last_mask) >> 3)
                              : (int64_t)0;
            nc = 1;
        }
    }
}

// Position of point j in the reference's tie order: its thread's rank among the
// bit-reversed thread ids times the points per thread, plus its turn within the thread.
__device__ __forceinline__ int fps_position_of_point(int j, const FpsLayout &L)
{
    const int t = j & (L.bs - 1);
    const int r = (int)(__builtin_bitreverse32((unsigned)t) >> (32 - L.log2_bs));
    return r * L.c + (j >> L.log2_bs);
}

// What one of these kernels leaves as a cloud's first index for the ones behind it.
constexpr int64_t FPS_ODD = -1;     // a coordinate is not finite: the plain loop has to do it
constexpr int64_t FPS_CLAIM = -2;   // the cloud looks as if in sampling order: to be checked
constexpr int FPS_CLAIM_MAX = 1024;

__device__ __forceinline__ int fps_max(int a, int b) { return a > b ? a : b; }
__device__ __forceinline__ int fps_min(int a, int b) { return a < b ? a : b; }

// The places of all cells of a 16^3 grid, by 256 x + 16 y + z. (Worked out for every point they took 150 operations,
// 13 us of the 612 at 8 x 16384 -> 4096 and 3 of the 155 at 16 x 4096 -> 1024.)
struct FpsCurve {
    unsigned short place[4096];
};
constexpr FpsCurve fps_make_curve()
{
    FpsCurve t{};
    for (unsigned i = 0; i < 4096u; ++i)
        t.place[i] = (unsigned short)tk_hilbert(i >> 8, (i >> 4) & 15u, i & 15u);
    return t;
}
__device__ constexpr FpsCurve fps_curve alignas(16) = fps_make_curve();

// Adds to a counter in LDS, lane by lane, and returns what it held before. (As an atomicAdd the
// compiler turns it into a scan over the lanes, for a handful of which it is.)
__device__ __forceinline__ int fps_lds_add(int *counter, int v)
{
    int before;
    const unsigned at = (unsigned)(size_t)(__attribute__((address_space(3))) int *)counter;
    asm volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)"
                 : "=v"(before)
                 : "v"(at), "v"(v)
                 : "memory");
    return before;
}

// Appends the lane's bit of a mask to a number: 2 bits + (mask >> lane & 1), in one instruction.
__device__ __forceinline__ unsigned fps_append(unsigned bits, unsigned long long mask)
{
    asm("v_addc_co_u32_e64 %0, vcc, %0, %0, %1" : "+v"(bits) : "s"(mask) : "vcc");
    return bits;
}

// Zero exactly if the lane's bits have none in common with the mask. (Of 64 bits compared at once, the
// comparison alone takes as long as all of this.)
__device__ __forceinline__ unsigned fps_common(unsigned long long bits, unsigned long long mask)
{
    unsigned some;
    asm("v_and_or_b32 %0, %1, %2, %3"
        : "=v"(some)
        : "v"((unsigned)(bits >> 32)), "s"((unsigned)(mask >> 32)), "v"((unsigned)bits & (unsigned)mask));
    return some;
}

// Width of a band for `target` points where one of width `was` held n. (Any number will do, as long as
// all waves have the same; a wave-uniform result.)
__device__ __forceinline__ int fps_band(int was, float target, int n)
{
    const float w = (float)was * (target * __builtin_amdgcn_rcpf((float)n));
    return __builtin_amdgcn_readfirstlane((int)__builtin_fmaxf(__builtin_fminf(w, 1e9f), 1.0f));
}

// fp32 kernel for clouds of up to 16384 points: dozens of selection steps per exchange between the
// waves, with the points laid out by region, so that an update only visits the points a new centre
// can reach.
//
// Band. With an upper bound `base` of all minima, the points whose running minimum lies above
// theta = base - step are listed in LDS, at most 64, a lane each; every other point is at or below
// theta. So as long as the steps' maxima stay above theta, the coming winners are found among the
// listed points alone: in order of (minimum, position), a listed point is a winner unless an earlier
// winner lies nearer to it than its minimum. Such a point falls to that distance, nearly always
// below theta (its neighbour in the same hole was taken); where it stays above, the list counts only
// down to that distance, `stop`, which takes theta's place. After the exchange nothing is above `stop`:
// the next `base`. The band's width follows the last one's (40 points are aimed at, 20 to 64 come):
// too many or none, and the points are listed again with another width, in two consecutive bands of
// that kind with the largest minimum looked for as well. 457 -> 139 exchanges at 16384 -> 4096, 155 -> 53
// at 4096 -> 1024, against a candidate from each of 128 groups of lanes and a list of sixteen.
//
// Judgement. Eight waves take eight listed points each and compare them with all 64 lanes: which
// come after, which of these are nearer than their minimum, a bit each, appended lane by lane with
// an add-with-carry. From the other waves' bits in LDS every wave then has, for its lane's point, the
// earlier points that would knock it out, and settles all of them in a few turns: a point none of whose
// opponents is undecided or a winner is a winner, one with a winner among them is out. (The list
// needs no order: a winner's turn is the number of winners before it.)
//
// Update. A winner with minimum v lowers minima only within sqrt(v) of itself, since no minimum is
// larger at its step. The prologue sorts the points along a Hilbert curve (a counting sort by cell in
// LDS) and cuts the sequence into NB NW regions; region R goes to wave R % NW as block R / NW of the
// lanes' registers (P / NB points per lane and block). A lane evaluates the canonical distance from
// its point to the box of every block of the wave - the same rounded operations as tk_dist2 on the per-axis
// gaps, each of which is monotone, so the result is a lower bound of the canonical distance to every point
// of the box - and a winner updates a block only if that bound is below v. Skipping is therefore
// exact. (Along a Morton curve, whose runs jump, a winner reached 6.9 of 64 blocks and the busiest wave
// had 22.8 of an exchange's visits; now 4.2 and 9.5.)
//
// Ties. Equal minima are ordered by the reference's positions (see the top of the file), looked up only
// where two listed minima are equal. Where more than 64 points share the largest minimum, the band is
// the part of them below a position that moves up. Lattices take many steps per exchange this way: 16 x
// 4096 -> 1024 on one of 9 x 9 x 9 points 0.35 -> 0.19 ms.
//
// What bounds it: one workgroup has one compute unit, and an exchange is a chain of short phases (clocks
// at 16 x 4096 -> 1024, 16 waves, of 6700 for 19 winners, of which shorter chains of instructions have since
// taken 250: listing 1100, judgement 1700, resolving and turns 800, update 1540 on average and 2050 in
// the slowest wave, with the boxes; the rest is waiting at the barriers, and 14 of 67 bands are listed
// again). Measured (us; before: a candidate per group; both
// with what runs behind them): 8 x 16384 -> 4096 1390-1450 -> 545, on a noisy sphere 1120-1200 -> 520,
// in clusters 1180-1330 -> 695; 16 x 8192 -> 2048 590 -> 275; 16 x 4096 -> 1024 285 -> 150; 16 x 2048 -> 512
// 160 -> 94; 1 x 1024 -> 512 120 -> 69; on lattices, copies and a line 0.2 to 0.9 of the time before.
// Tried: listing up to 256 and judging the upper 64 (0 to 5 % faster up to 8192 points, 4 % slower
// at 16384, lattices 10 % slower), aiming at 28, 34, 56 or 80 points, blocks of half and twice the
// size and half as many waves with twice the points (all slower by 2 to 20 % at the sizes where another
// instance is used), a point's names and the loop's boxes kept in registers (they went to scratch: 2.1 times the
// time at 16384).
//
// A cloud that is itself a farthest point sample, in sampling order from its point 0 (the next level
// of a PointNet++ encoder), has 0, 1, 2, ... as its answer. Where point 1 is the point farthest from
// point 0, point 2 the one farthest from both and at most 1024 samples are wanted, this kernel
// only leaves the claim, which fps_claim_minima_kernel and fps_settle_kernel_f32 test with the whole
// chip; the latter writes the answer, or does the work (LAST) if the claim was wrong.
// (A cloud in random order passes the test of point 1 once in n, and then takes twice the time: with that
// test alone 256 x 2048 -> 512 took 330 us for 177 in one batch of eight. Point 2 is looked at behind it.)
template <int P, int NW, int NB, bool SOA, bool LAST>
__device__ __forceinline__ void fps_band(const float *__restrict__ pts, int64_t *__restrict__ out,
                                           const FpsLayout &L, bool claims)
{
    constexpr int NT = NW * TK_WAVE, PB = P / NB, S = NT * P, RS = TK_WAVE * PB;
    constexpr int LIST = TK_WAVE;                   // points judged at once, a lane each
    constexpr int QUAD = P < 4 ? P : 4;
    constexpr float TARGET = 40.0f;                 // points a band is meant to hold
    constexpr int NJ = NW < 8 ? NW : 8;             // waves that judge
    constexpr int RJ = TK_WAVE / NJ;                // points for which each of them does
    constexpr int RJ_LOG2 = RJ == 8 ? 3 : 4;
    using Piece = typename std::conditional<RJ == 8, unsigned char, unsigned short>::type;
    struct Relation {  // of a listed point to the others, a bit each
        Piece before[NJ];  // is before it
        Piece hit[NJ];     // and nearer to it than its minimum
    };
    constexpr int CELLS = 4096;                     // 16^3 cells for the sort
    static_assert((P & (P - 1)) == 0 && P % NB == 0 && (NW & (NW - 1)) == 0 && NW >= 4, "shape");
    static_assert(CELLS % NT == 0 && S < (1 << 19) && S >= 8 * LIST && P % QUAD == 0, "sort");
    constexpr int F32_NEG1 = (int)0xbf800000;
    extern __shared__ __align__(16) unsigned char fps_band_lds[];
    unsigned *const keys = reinterpret_cast<unsigned *>(fps_band_lds);  // [S] points, sorted
    unsigned *const cnt = keys + S;                                       // [CELLS + 1]
    __shared__ float4 s_cand[LIST + 1];  // the band's points: x, y, z, running minimum (bits)
    __shared__ int s_name[LIST + 1];     // which points those are
    __shared__ __align__(16) Relation s_rel[LIST];
    __shared__ int s_count[3], s_stop[3], s_most[3], s_step;
    __shared__ float s_red[NW][8];

    const int tid = threadIdx.x;
    const int lane = tid & (TK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE);
    const float INF = __builtin_huge_valf();

    float x[P], y[P], z[P];
    int t[P];  // running minimum of point p (bits)
    // what a point goes by outside its lane: its sorted rank. Block q, turn u of a lane holds
    // rank (q * NW + wave) * RS + u * 64 + lane.
    auto name_of = [&](int in_lane, int p) {
        return ((p / PB) * NW + wave) * RS + (p % PB) * TK_WAVE + in_lane;
    };
    auto point_of = [&](int name) { return (int)keys[name]; };
    // ---- bounding box of the cloud, whether it is finite, and how far from point 0 it reaches ----
    float lo[3] = {INF, INF, INF}, hi[3] = {-INF, -INF, -INF};
    const float p0[3] = {fps_coord<SOA>(pts, L.n, 0, 0), fps_coord<SOA>(pts, L.n, 0, 1),
                         fps_coord<SOA>(pts, L.n, 0, 2)};
    float far = 0.0f;
    float zero = 0.0f;
    float own[3][P];  // point tid + k * NT (beyond the cloud: its last point), read coalesced
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int e = fps_min(tid + k * NT, L.n - 1);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            own[a][k] = fps_coord<SOA>(pts, L.n, e, a);
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = __builtin_fminf(lo[a], own[a][k]);
            hi[a] = __builtin_fmaxf(hi[a], own[a][k]);
            zero = __builtin_fmaf(own[a][k], 0.0f, zero);  // (NaN once one is not finite)
        }
        far = __builtin_fmaxf(far, tk_dist2<float>(own[0][k], own[1][k], own[2][k], p0[0], p0[1],
                                                   p0[2]));
    }
    far = wave_max<float>(far);
    const bool odd = __builtin_amdgcn_ballot_w64(!(zero == 0.0f)) != 0ull;
    float ends[6] = {-lo[0], -lo[1], -lo[2], hi[0], hi[1], hi[2]};
    tk_wave_max_six<64>(ends);
    if (lane == TK_WAVE - 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            s_red[wave][a] = -ends[a];
            s_red[wave][3 + a] = ends[3 + a];
        }
        s_red[wave][6] = odd ? -1.0f : far;
    }
    // (the table where the list comes later, if there is room)
    constexpr bool NEAR = S * 4 >= (int)sizeof(FpsCurve);
    if constexpr (NEAR)
        for (int i = tid; i < (int)sizeof(FpsCurve) / 16; i += NT)
            reinterpret_cast<uint4 *>(fps_band_lds)[i] = reinterpret_cast<const uint4 *>(&fps_curve)[i];
    const unsigned short *const curve =
        NEAR ? reinterpret_cast<const unsigned short *>(fps_band_lds) : fps_curve.place;
    for (int i = tid; i <= CELLS; i += NT)
        cnt[i] = 0u;
    if (tid < 3)
        s_count[tid] = s_stop[tid] = s_most[tid] = 0;
    __syncthreads();
    float reached = 0.0f;
    bool any_odd = false;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        reached = __builtin_fmaxf(reached, s_red[w][6]);
        any_odd |= s_red[w][6] < 0.0f;
    }
    if constexpr (!LAST) {
        const float p1[3] = {fps_coord<SOA>(pts, L.n, 1, 0), fps_coord<SOA>(pts, L.n, 1, 1),
                             fps_coord<SOA>(pts, L.n, 1, 2)};
        bool claim = claims && !any_odd &&
                     tk_dist2<float>(p1[0], p1[1], p1[2], p0[0], p0[1], p0[2]) >= reached;
        if (claim) {  // uniform over the workgroup: step 2 has taken the farthest from points 0 and 1
            const auto from_both = [&](float px, float py, float pz) {
                return __builtin_fminf(tk_dist2<float>(px, py, pz, p0[0], p0[1], p0[2]),
                                       tk_dist2<float>(px, py, pz, p1[0], p1[1], p1[2]));
            };
            far = 0.0f;
#pragma unroll
            for (int k = 0; k < P; ++k)
                far = __builtin_fmaxf(far, from_both(own[0][k], own[1][k], own[2][k]));
            far = wave_max<float>(far);
            if (lane == 0)
                s_red[wave][7] = far;
            __syncthreads();
            float both = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w)
                both = __builtin_fmaxf(both, s_red[w][7]);
            claim = from_both(fps_coord<SOA>(pts, L.n, 2, 0), fps_coord<SOA>(pts, L.n, 2, 1),
                              fps_coord<SOA>(pts, L.n, 2, 2)) >= both;
        }
        if (any_odd || claim) {  // uniform over the workgroup
            if (tid == 0) {
                out[0] = any_odd ? FPS_ODD : FPS_CLAIM;
                out[1] = 0;
            }
            return;
        }
    }
    float origin[3], scale[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float l = INF, h = -INF;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            l = __builtin_fminf(l, s_red[w][a]);
            h = __builtin_fmaxf(h, s_red[w][3 + a]);
        }
        origin[a] = l;
        const float extent = h - l;
        scale[a] = extent > 0.0f ? 15.99f / extent : 0.0f;  // also 0 for NaN / inf extents
    }

    // ---- the points in the order of their cells along the curve; slots beyond the cloud
    // last. A counting sort: any order that keeps neighbours together is a valid layout, so 16
    // steps per axis are enough and the order within a cell is whatever the atomics give. ----
    unsigned where[P];  // cell, and the point's turn within it from bit 13
#pragma unroll
    for (int k = 0; k < P; ++k) {
        unsigned cell = CELLS;
        if (tid + k * NT < L.n) {
            unsigned at = 0u;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float f = (own[a][k] - origin[a]) * scale[a];
                // (a NaN or an out-of-range value lands in cell 0 or 15)
                at = 16u * at + (unsigned)(int)__builtin_fminf(__builtin_fmaxf(f, 0.0f), 15.0f);
            }
            cell = curve[at];
        }
        where[k] = cell | (atomicAdd(&cnt[cell], 1u) << 13);
    }
    __syncthreads();
    {
        // counts -> first positions: a lane sums its run of counters, the waves scan the sums
        constexpr int RUN = CELLS / NT;
        unsigned c[RUN], mine = 0u;
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            c[i] = cnt[tid * RUN + i];
            mine += c[i];
        }
        unsigned incl = mine;
#pragma unroll
        for (int o = 1; o < TK_WAVE; o <<= 1) {
            const unsigned up = (unsigned)__shfl_up((int)incl, o);
            incl += lane >= o ? up : 0u;
        }
        if (lane == TK_WAVE - 1)
            s_red[wave][7] = __builtin_bit_cast(float, incl);
        __syncthreads();
        unsigned start = incl - mine;
        for (int w = 0; w < wave; ++w)
            start += __builtin_bit_cast(unsigned, s_red[w][7]);
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            cnt[tid * RUN + i] = start;
            start += c[i];
        }
        if (tid == 0)
            cnt[CELLS] = (unsigned)L.n;  // the slots beyond the cloud follow its points
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < P; ++k)
        where[k] = cnt[where[k] & 0x1fffu] + (where[k] >> 13);  // the point's sorted rank
    __syncthreads();
    // ---- this lane's points: block q, turn u <-> sorted rank (q*NW + wave) * RS + u*64 + lane.
    // The coordinates travel through LDS, x and y first, then z with the list of points, which
    // stays (fetched from memory by rank they are 48 gathers of 64 cache lines per wave). ----
    float *const plane0 = reinterpret_cast<float *>(keys), *const plane1 = plane0 + S;
#pragma unroll
    for (int k = 0; k < P; ++k) {
        plane0[where[k]] = own[0][k];
        plane1[where[k]] = own[1][k];
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        x[p] = plane0[name_of(lane, p)];
        y[p] = plane1[name_of(lane, p)];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < P; ++k) {
        keys[where[k]] = (unsigned)(tid + k * NT);
        plane1[where[k]] = own[2][k];
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        z[p] = plane1[name_of(lane, p)];
    }
    // ---- minima after point 0, boxes of the wave's blocks (an empty block gets an empty box: never
    // reached), wave-uniform ----
    float box[NB][6];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        float reach[6] = {-INF, -INF, -INF, -INF, -INF, -INF};  // -lowest, highest
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int p = q * PB + u;
            const bool ok = name_of(lane, p) < L.n;  // (the slots beyond the cloud come last)
            const float v[3] = {x[p], y[p], z[p]};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                reach[a] = __builtin_fmaxf(reach[a], ok ? -v[a] : -INF);
                reach[3 + a] = __builtin_fmaxf(reach[3 + a], ok ? v[a] : -INF);
            }
            const float d = tk_dist2<float>(x[p], y[p], z[p], p0[0], p0[1], p0[2]);
            t[p] = ok ? __builtin_bit_cast(int, d) : F32_NEG1;
        }
        tk_wave_max_six<64>(reach);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            box[q][a] = -read_lane(reach[a], TK_WAVE - 1);
            box[q][3 + a] = read_lane(reach[3 + a], TK_WAVE - 1);
        }
    }
    __syncthreads();  // plane1 is read
    // The picks by name, in order, where the sort had its counters (k <= n <= S).
    int *const order = reinterpret_cast<int *>(plane1);
    int base = __builtin_bit_cast(int, reached);  // no minimum is above it
    int step = 1 << 19;                           // width of the band below it, in steps of a float
    // With `tied` the band is part of the points whose minimum is `base` itself: those at positions
    // before tie_end (and from tie_from on, there are none before it).
    bool tied = false;
    int tie_from = 0, tie_end = 0, tie_step = S / 8;
    int wide = step;  // the last band that was not of equals

    const int own_slot = (lane >> RJ_LOG2) + NJ * (lane & (RJ - 1));  // lane 8 w + i has candidate w + 8 i
    const auto after = [](int turn) { return turn == 2 ? 0 : turn + 1; };
    int it = 1, n = 0, turn = 0;  // (turn: which of three counters)
    while (it < L.k) {  // (uniform over the workgroup, as is all of this state)
        // ---- the points of the band; anew with another band if they are too many or none ----
        int theta;
        int crowd = 1 << 20;
        bool again = false;  // (then the largest minimum is looked for as well)
        float4 C;
        int my_name;
        for (;; turn = after(turn), again = true) {
            theta = tied ? base - 1 : fps_max(base - step, 0);
            int *const count = &s_count[turn];
            if (tid == 0)  // (their last readers are two barriers back)
                s_count[after(turn)] = s_stop[after(turn)] = s_most[after(turn)] = 0;
            int first = wave * RS + lane;  // a point's name is this and a constant
            asm volatile("" : "+v"(first));  // (added where it is wanted, not kept in P registers)
            const auto enlist = [&](int p, int &at) {
                const int to = fps_min(at, LIST);  // (what is too much goes to a spare place)
                s_cand[to] = make_float4(x[p], y[p], z[p], __builtin_bit_cast(float, t[p]));
                s_name[to] = first + (p / PB) * NW * RS + (p % PB) * TK_WAVE;
                ++at;
            };
            if (__builtin_expect(!tied, 1)) {  // uniform
                int upto[P / QUAD], mine = 0;  // how many there are in the lane's first points
#pragma unroll
                for (int g = 0; g < P / QUAD; ++g) {
#pragma unroll
                    for (int p = g * QUAD; p < (g + 1) * QUAD; ++p)
                        mine += t[p] > theta ? 1 : 0;
                    upto[g] = mine;
                }
                if (mine > 0) {
                    int at = fps_lds_add(count, mine);
#pragma unroll
                    for (int g = 0; g < P / QUAD; ++g) {
                        if (upto[g] > (g > 0 ? upto[g - 1] : 0)) {
#pragma unroll
                            for (int p = g * QUAD; p < (g + 1) * QUAD; ++p) {
                                if (t[p] > theta)
                                    enlist(p, at);
                            }
                        }
                    }
                }
            } else {
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    if (t[p] > theta &&
                        fps_position_of_point(point_of(first + (p / PB) * NW * RS + (p % PB) * TK_WAVE), L) < tie_end) {
                        int at = fps_lds_add(count, 1);
                        enlist(p, at);
                    }
                }
            }
            if (again && !tied) {  // uniform
                int most = t[0];
#pragma unroll
                for (int p = 1; p < P; ++p)
                    most = fps_max(most, t[p]);
                most = wave_max_i32(fps_max(most, 0));
                if (lane == 0)
                    atomicMax(&s_most[turn], most);
            }
            __syncthreads();
            const int listed = *count;
            C = s_cand[own_slot];  // (requested before the count is looked at)
            my_name = s_name[own_slot];
            n = __builtin_amdgcn_readfirstlane(listed);
            if ((unsigned)(n - 1) < (unsigned)LIST)
                break;
            if (n == 0) {
                if (tied) {  // none before tie_end
                    if (tie_end < S) {
                        tie_step = 2 * tie_step;
                        tie_from = tie_end;
                        tie_end = fps_min(tie_from + tie_step, S);
                    } else {
                        tied = false;
                        base -= 1;
                        step = wide;
                    }
                } else {
                    if (theta == 0)
                        break;  // no point lies away from the chosen set, and none will
                    base = again ? __builtin_amdgcn_readfirstlane(s_most[turn]) : theta;
                    step = fps_min(2 * step, 1 << 24);
                }
            } else if (tied) {  // (positions differ: LIST of them hold no more points)
                tie_step = (tie_end - tie_from) >> 1;
                tie_end = tie_from + tie_step;
            } else if (base - theta == 1) {  // too many points share the largest minimum
                tied = true;
                tie_from = 0;
                tie_end = fps_min(tie_step, S);
            } else {
                step = base - theta;
                if (again)
                    base = __builtin_amdgcn_readfirstlane(s_most[turn]);
                // (where a narrower band has not made them fewer, they are equal)
                step = 4 * n > 3 * crowd ? 1 : fps_band(step, TARGET, n);
                crowd = n;
            }
        }
        if (n == 0)
            break;
        const auto next_step = [&] {
            const int was = base - theta;
            const int w = fps_max(fps_min(fps_max(fps_band(was, TARGET, n), was >> 1), 2 * was), 1);
            return fps_min(w, 1 << 24);
        };
        if (NW > NJ && wave == NW - 1 && !tied) {  // uniform; it has nothing to judge
            const int w = next_step();
            if (lane == 0)
                s_step = w;
        }
        const int v = own_slot < n ? __builtin_bit_cast(int, C.w) : -1;
        if (wave < NJ) {
            // wave w relates the candidates of lanes RJ w .. to all of them
            unsigned hits = 0u, befores = 0u;
            int over = 0;  // the largest distance to which a candidate falls
            int pos = -1;
            bool have_pos = false;
            const int rows = (n - wave + NJ - 1) / NJ;
            const auto relate = [&](auto pair, int r) {  // the candidates of lanes r and, with pair, r + 1
                constexpr int R = decltype(pair)::value;
                float d[R];
                int rv[R];
                unsigned long long after[R], hit[R], same[R];
                int equals = 0;
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    rv[j] = read_lane(v, r + j);
                    d[j] = tk_dist2<float>(C.x, C.y, C.z, read_lane(C.x, r + j), read_lane(C.y, r + j),
                                           read_lane(C.z, r + j));
                    after[j] = __builtin_amdgcn_ballot_w64(rv[j] > v);
                    same[j] = __builtin_amdgcn_ballot_w64(rv[j] == v);
                    equals += __builtin_popcountll(same[j]);
                }
                if (__builtin_expect(equals != R, 0)) {  // uniform
                    if (!have_pos) {
                        pos = fps_position_of_point(point_of(v >= 0 ? my_name : 0), L);
                        have_pos = true;
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j)
                        after[j] |= same[j] & __builtin_amdgcn_ballot_w64(read_lane(pos, r + j) < pos);
                }
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    hit[j] = after[j] & __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int, d[j]) < v);
                    over = fps_max(over, __builtin_amdgcn_inverse_ballot_w64(hit[j]) ? __builtin_bit_cast(int, d[j]) : 0);
                }
#pragma unroll
                for (int j = R - 1; j >= 0; --j) {
                    befores = fps_append(befores, after[j]);
                    hits = fps_append(hits, hit[j]);
                }
            };
            if (rows & 1)  // uniform
                relate(std::integral_constant<int, 1>{}, RJ * wave + rows - 1);
#pragma unroll 1
            for (int i = (rows & ~1) - 2; i >= 0; i -= 2)
                relate(std::integral_constant<int, 2>{}, RJ * wave + i);
            s_rel[lane].before[wave] = (Piece)befores;
            s_rel[lane].hit[wave] = (Piece)hits;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(over > theta) != 0ull, 0)) {  // uniform
                over = wave_max_i32(over);
                if (lane == 0)
                    atomicMax(&s_stop[turn], over);
            }
        }
        __syncthreads();
        const ulonglong2 rel = *reinterpret_cast<const ulonglong2 *>(&s_rel[lane]);
        const unsigned long long before = rel.x, hit = rel.y;
        const int stop = __builtin_amdgcn_readfirstlane(fps_max(theta, s_stop[turn]));
        const int its_step = s_step;
        unsigned long long open = __builtin_amdgcn_ballot_w64(v >= 0), winners = 0ull;
        while (open != 0ull) {  // (the first of the open ones is decided in every turn)
            const unsigned long long may = open | winners;
            const unsigned long long won = __builtin_amdgcn_ballot_w64(fps_common(hit, may) == 0u) & open;
            winners |= won;
            const unsigned long long lost = __builtin_amdgcn_ballot_w64(fps_common(hit, winners) != 0u) & open;
            open &= ~(won | lost);
        }
        winners &= __builtin_amdgcn_ballot_w64(v > stop);
        // ---- their turns, and the minima they lower ----
        if (wave == NW - 1) {  // uniform
            unsigned long long mine = before;
            asm volatile("" : "+v"(mine));  // (the others are not to work it out as well)
            const int at = it + __builtin_popcountll(mine & winners);
            if (__builtin_amdgcn_inverse_ballot_w64(winners) && at < L.k)
                order[at] = my_name;
        }
        it += __builtin_popcountll(winners);
        if (!tied) {
            step = NW > NJ ? __builtin_amdgcn_readfirstlane(its_step) : next_step();
            wide = fps_max(step, wide >> 1);
            base = stop;
        } else {
            tie_step = n < LIST / 2 ? fps_min(2 * tie_step, S) : tie_step;
            tie_from = tie_end;
            tie_end = fps_min(tie_from + tie_step, S);
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const float gx = __builtin_fmaxf(__builtin_fmaxf(box[q][0] - C.x, C.x - box[q][3]), 0.0f);
            const float gy = __builtin_fmaxf(__builtin_fmaxf(box[q][1] - C.y, C.y - box[q][4]), 0.0f);
            const float gz = __builtin_fmaxf(__builtin_fmaxf(box[q][2] - C.z, C.z - box[q][5]), 0.0f);
            const float bound = __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
            unsigned long long todo = __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int, bound) < v) & winners;
            if (todo != 0ull) {  // uniform
                if (__builtin_popcountll(todo) & 1) {  // uniform
                    const int l = __builtin_ctzll(todo);
                    const float sx = read_lane(C.x, l), sy = read_lane(C.y, l), sz = read_lane(C.z, l);
#pragma unroll
                    for (int u = 0; u < PB; ++u) {
                        const int p = q * PB + u;
                        const float d = tk_dist2<float>(x[p], y[p], z[p], sx, sy, sz);
                        t[p] = fps_min(t[p], __builtin_bit_cast(int, d));
                    }
                    todo &= todo - 1;
                }
                while (todo != 0ull) {  // two at a time
                    const int l = __builtin_ctzll(todo);
                    const float sx = read_lane(C.x, l), sy = read_lane(C.y, l), sz = read_lane(C.z, l);
                    todo &= todo - 1;
                    const int h = __builtin_ctzll(todo);
                    const float hx = read_lane(C.x, h), hy = read_lane(C.y, h), hz = read_lane(C.z, h);
                    todo &= todo - 1;
#pragma unroll
                    for (int u = 0; u < PB; ++u) {
                        const int p = q * PB + u;
                        const float d = tk_dist2<float>(x[p], y[p], z[p], sx, sy, sz);
                        const float e = tk_dist2<float>(x[p], y[p], z[p], hx, hy, hz);
                        t[p] = fps_min(fps_min(t[p], __builtin_bit_cast(int, d)),
                                       __builtin_bit_cast(int, e));
                    }
                }
            }
        }
        turn = after(turn);
    }
    __syncthreads();
    // (after the last point that lies away from the chosen ones the previous choice is repeated)
    const int64_t again = it > 1 ? (int64_t)point_of(order[fps_min(it, L.k) - 1]) : 0;
    for (int i = tid; i < L.k; i += NT)
        out[i] = i == 0 ? 0 : i < it ? (int64_t)point_of(order[i]) : again;
}

template <int P, int NW, int NB, bool SOA>
__global__ __launch_bounds__(NW * 64) void fps_band_kernel_f32(const float *__restrict__ points,
                                                                 int64_t *__restrict__ index,
                                                                 FpsLayout L, bool claims)
{
    fps_band<P, NW, NB, SOA, false>(points + (int64_t)blockIdx.x * L.n * 3,
                                      index + (int64_t)blockIdx.x * L.k, L, claims);
}

// A claim that a cloud's first k points, in this order, are its farthest point sample: step s takes point s
// exactly if no point has a larger running minimum after the centres 0 .. s - 1, nor an equal one at a
// lower position. The minimum of point s itself at that time, v_s, is the threshold, worked out by a first
// kernel into the index row, which nobody else needs yet; fps_settle_kernel_f32 compares. Both read the centres at
// uniform addresses and cut them into stretches, a wave each. A cloud's workgroups take its groups of 64 points in
// turn. 8 x 4096 -> 1024: 333 us of sampling before, 36 us in all.
constexpr int FPS_CLAIM_PARTS = 16;

template <bool SOA>
__global__ __launch_bounds__(1024) void fps_claim_minima_kernel(const float *__restrict__ points,
                                                                int64_t *__restrict__ index,
                                                                FpsLayout L, int slices)
{
    const int b = blockIdx.x / slices;
    const float *__restrict__ pts = points + (int64_t)b * L.n * 3;
    int64_t *__restrict__ out = index + (int64_t)b * L.k;
    if (out[0] != FPS_CLAIM)  // uniform over the workgroup
        return;
    __shared__ float s_min[FPS_CLAIM_PARTS][TK_WAVE];
    const int lane = threadIdx.x & (TK_WAVE - 1);
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
    for (int first = blockIdx.x % slices * TK_WAVE; first < L.k; first += slices * TK_WAVE) {
        const int s = first + lane, me = s < L.k ? s : L.k - 1;
        const float x = fps_coord<SOA>(pts, L.n, me, 0), y = fps_coord<SOA>(pts, L.n, me, 1),
                    z = fps_coord<SOA>(pts, L.n, me, 2);
        const int end = fps_min(first + TK_WAVE, L.k);  // centres below end can matter
        const int step = (end + FPS_CLAIM_PARTS - 1) / FPS_CLAIM_PARTS;
        float m = __builtin_huge_valf();
#pragma unroll 4
        for (int i = part * step; i < fps_min((part + 1) * step, end); ++i) {
            const float d = tk_dist2<float>(x, y, z, fps_coord<SOA>(pts, L.n, i, 0),
                                            fps_coord<SOA>(pts, L.n, i, 1), fps_coord<SOA>(pts, L.n, i, 2));
            m = i < s ? __builtin_fminf(m, d) : m;
        }
        s_min[part][lane] = m;
        __syncthreads();
        if (part == 0 && s > 0 && s < L.k) {
#pragma unroll
            for (int w = 1; w < FPS_CLAIM_PARTS; ++w)
                m = __builtin_fminf(m, s_min[w][lane]);
            out[s] = (int64_t)__builtin_bit_cast(int, m);
        }
        __syncthreads();  // (the next turn writes s_min)
    }
}

// Whether a claim fails on one of the workgroup's points (of one thread's, in that thread).
template <int NW, bool SOA>
__device__ __forceinline__ bool fps_claim_fails(const float *__restrict__ pts, const int64_t *out,
                                                const FpsLayout &L, int slice, int slices)
{
    // Centres that a wave takes at a time. Their distances stay in registers until the minima over the waves
    // before it are there, and the differences to the thresholds run into one maximum: worked out twice, and
    // compared step by step, the check took 35 us at 8 x 4096 -> 1024 and 5 more for the launch behind it, both
    // now 24.
    constexpr int C = 32;
    __shared__ __align__(16) float s_v[FPS_CLAIM_MAX + C * NW];  // [i]: v of step i + 1, which follows centre i
    __shared__ float s_min[2][NW][TK_WAVE];
    const int lane = threadIdx.x & (TK_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TK_WAVE);
    const int centres = L.k - 1;
    bool bad = false;
    for (int i = threadIdx.x; i < FPS_CLAIM_MAX + C * NW; i += NW * TK_WAVE) {
        const float v = i < centres ? __builtin_bit_cast(float, (int)out[i + 1]) : __builtin_huge_valf();
        bad |= !(v > 0.0f && (v < __builtin_huge_valf() || i >= centres));
        s_v[i] = v;
    }
    __syncthreads();
    int turn = 0;
    for (int first = slice * TK_WAVE; first < L.n; first += slices * TK_WAVE) {
        const int j = first + lane, me = j < L.n ? j : L.n - 1;
        const float x = fps_coord<SOA>(pts, L.n, me, 0), y = fps_coord<SOA>(pts, L.n, me, 1),
                    z = fps_coord<SOA>(pts, L.n, me, 2);
        float before = __builtin_huge_valf();  // the minimum over the centres up to this turn's
        for (int start = 0; start < centres; start += C * NW, turn ^= 1) {
            const int from = start + wave * C;
            float m[C];
            const auto minima = [&](auto whole) {  // (whole: at addresses that the compiler sees are side by side)
#pragma unroll
                for (int u = 0; u < C; ++u) {  // (beyond the last centre v is infinite)
                    const int i = whole ? from + u : fps_min(from + u, centres - 1);
                    const float d = tk_dist2<float>(x, y, z, fps_coord<SOA>(pts, L.n, i, 0),
                                                    fps_coord<SOA>(pts, L.n, i, 1), fps_coord<SOA>(pts, L.n, i, 2));
                    m[u] = u ? __builtin_fminf(m[u ? u - 1 : 0], d) : d;
                }
            };
            if (from + C <= centres)
                minima(std::true_type());
            else
                minima(std::false_type());
            s_min[turn][wave][lane] = m[C - 1];
            __syncthreads();
            float here = before;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float o = s_min[turn][w][lane];
                here = w < wave ? __builtin_fminf(here, o) : here;
                before = __builtin_fminf(before, o);
            }
            float over = -1.0f;  // the largest minimum less its threshold
            const auto compare = [&](auto meets) {
#pragma unroll
                for (int u = 0; u < C; ++u) {
                    const float d = __builtin_fminf(m[u], here) - s_v[from + u];
                    over = __builtin_fmaxf(over, meets && me == from + u + 1 ? -1.0f : d);
                }
            };
            if (first <= from + C && from < first + TK_WAVE)  // a point of the group meets its own v here
                compare(std::true_type());
            else
                compare(std::false_type());
            bad |= over > 0.0f;
            if (__builtin_amdgcn_ballot_w64(over == 0.0f) != 0ull)  // a tie
                for (int i = from; i < fps_min(from + C, centres); ++i) {
                    here = __builtin_fminf(here, tk_dist2<float>(x, y, z, fps_coord<SOA>(pts, L.n, i, 0),
                                                                 fps_coord<SOA>(pts, L.n, i, 1),
                                                                 fps_coord<SOA>(pts, L.n, i, 2)));
                    const float v = s_v[i];
                    if (here == v && me != i + 1)
                        bad |= fps_position_of_point(me, L) < fps_position_of_point(i + 1, L);
                }
        }
    }
    return bad;
}

// Behind the band kernel: claims are checked, the clouds that it has left done, and the coordinates follow the
// indices. A cloud's workgroups share the check and the copying; what has to be done by one of them is done by
// the last one through. Its turn is counted, with who has found the claim wrong from bit 16, in the upper half of
// out[1], which is zero until then (out[1] holds v_1, a float); nobody waits for anybody, and what a cloud is
// in for is read from out[0] before the turn is taken, so only the last one changes it, after all have read it.
// (Against a launch for the check and one for the rest, us: 4 x 1024 -> 512 75.3, 74.0; 8 x 16384 -> 1024 304,
// 300, where one workgroup copied a cloud's coordinates; a claim that fails late 16 x 4096 -> 1024 249, 255, and 175
// with the shorter exchanges since.)
template <int P, int NW, int NB, bool SOA>
__global__ __launch_bounds__(NW * 64) void fps_settle_kernel_f32(const float *__restrict__ points,
                                                                 int64_t *__restrict__ index,
                                                                 float *__restrict__ sampled,
                                                                 FpsLayout L, int slices)
{
    constexpr int NT = NW * TK_WAVE;
    const int b = blockIdx.x / slices;
    int slice = blockIdx.x % slices, of = slices;
    const float *__restrict__ pts = points + (int64_t)b * L.n * 3;
    int64_t *out = index + (int64_t)b * L.k;
    const int64_t left = out[0];  // uniform over the workgroup
    if (left < 0) {
        __shared__ unsigned s_turn;
        bool bad = false;
        if (left == FPS_CLAIM)
            bad = fps_claim_fails<NW, SOA>(pts, out, L, slice, slices);
        bad = __syncthreads_or(bad);
        if (threadIdx.x == 0)
            s_turn = __hip_atomic_fetch_add(reinterpret_cast<unsigned *>(out + 1) + 1, bad ? 0x10001u : 1u,
                                            __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const unsigned turn = s_turn;
        if ((turn & 0xffffu) != (unsigned)(slices - 1))
            return;
        if (left == FPS_ODD)
            fps_plain<float, P, NT, SOA>(pts, out, L);
        else if (bad || turn >> 16)
            fps_band<P, NW, NB, SOA, true>(pts, out, L, false);
        else
            for (int i = threadIdx.x; i < L.k; i += NT)
                out[i] = (int64_t)i;
        __syncthreads();
        slice = 0;
        of = 1;
    }
    if (sampled) {
        float *__restrict__ so = sampled + (int64_t)b * L.k * 3;
        for (int i = slice * NT + threadIdx.x; i < L.k; i += of * NT) {
            const int64_t j = out[i];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                so[SOA ? (int64_t)a * L.k + i : (int64_t)i * 3 + a] = fps_coord<SOA>(pts, L.n, j, a);
        }
    }
}

// Clouds that do not fit in one workgroup's registers: every selection step is one
// launch of many workgroups per cloud. Step s first works out the point chosen by step
// s - 1 from the candidates that step's workgroups left in the workspace (every workgroup
// redoes this small reduction itself), then updates the running minima of its own slice
// of the cloud for that centre, streaming coordinates and minima through coalesced
// loads, and leaves its own candidate for step s + 1. The kernel boundary is the
// cross-workgroup barrier; nothing waits inside a kernel.
//
// Points are visited in index order; the reference's tie order is restored by comparing
// positions (see the top of the file) whenever two minima are equal.
template <typename T> struct FpsWideArgs {
    const T *points;     // [B, n, 3] or [B, 3, n]
    int64_t *index;      // [B, k]
    T *min_dist;         // [B, n]
    T *cand_val;         // [2, B, groups]: largest running minimum of a workgroup's slice
    int *cand_pos;       // [2, B, groups]: its position
    int *chosen;         // [2, B]: the point the previous step used as centre
    int groups;          // workgroups per cloud
    int slice;           // points per workgroup
    int batch;           // B
};

// (value, position) pairs ordered by larger value, then lower position.
template <typename T>
__device__ __forceinline__ void fps_keep_better(T &val, int &pos, T oval, int opos)
{
    const bool take = oval > val || (oval == val && opos < pos);
    val = take ? oval : val;
    pos = take ? opos : pos;
}

template <typename T, int NT>
__device__ __forceinline__ void fps_block_best(T &val, int &pos, T *s_val, int *s_pos)
{
    constexpr int NW = NT / TK_WAVE;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const T oval = __shfl_xor(val, o);
        const int opos = __shfl_xor(pos, o);
        fps_keep_better<T>(val, pos, oval, opos);
    }
    __syncthreads();  // the arrays may still be read from an earlier call
    if ((threadIdx.x & (TK_WAVE - 1)) == 0) {
        s_val[threadIdx.x / TK_WAVE] = val;
        s_pos[threadIdx.x / TK_WAVE] = pos;
    }
    __syncthreads();
    val = s_val[0];
    pos = s_pos[0];
#pragma unroll
    for (int w = 1; w < NW; ++w)
        fps_keep_better<T>(val, pos, s_val[w], s_pos[w]);
}

template <typename T, int NT, bool SOA>
__global__ __launch_bounds__(NT) void fps_wide_step_kernel(FpsWideArgs<T> a, FpsLayout L,
                                                           int step)
{
    __shared__ T s_val[NT / TK_WAVE];
    __shared__ int s_pos[NT / TK_WAVE];
    const int tid = threadIdx.x;
    const int g = blockIdx.x, b = blockIdx.y;
    const T *__restrict__ pts = a.points + (int64_t)b * L.n * 3;
    constexpr int NO_POS = 0x7fffffff;

    // ---- the centre of this step: what step - 1 selected ----
    int centre = 0;
    if (step > 1) {
        const int from = (step - 1) & 1;
        const T *cv = a.cand_val + ((int64_t)from * a.batch + b) * a.groups;
        const int *cp = a.cand_pos + ((int64_t)from * a.batch + b) * a.groups;
        T val = (T)0;
        int pos = NO_POS;
        for (int i = tid; i < a.groups; i += NT)
            fps_keep_better<T>(val, pos, cv[i], cp[i]);
        fps_block_best<T, NT>(val, pos, s_val, s_pos);
        // Nothing above zero: no point lies away from the chosen set and the previous
        // choice is emitted again, as the reference does.
        centre = val > (T)0 ? fps_point_of_position(pos, L) : a.chosen[(int64_t)from * a.batch + b];
    }
    if (g == 0 && tid == 0) {
        a.index[(int64_t)b * L.k + (step - 1)] = (int64_t)centre;
        a.chosen[(int64_t)(step & 1) * a.batch + b] = centre;
    }
    if (step >= L.k)  // the last launch only records the last choice
        return;

    // ---- update this workgroup's slice, keep its best candidate ----
    const T cx = fps_coord<SOA>(pts, L.n, centre, 0), cy = fps_coord<SOA>(pts, L.n, centre, 1),
            cz = fps_coord<SOA>(pts, L.n, centre, 2);
    T *__restrict__ md = a.min_dist + (int64_t)b * L.n;
    const int j0 = g * a.slice;
    const int j1 = (j0 + a.slice < L.n) ? j0 + a.slice : L.n;
    T best = (T)0;
    int bpos = NO_POS;
    for (int j = j0 + tid; j < j1; j += NT) {
        T x, y, z;
        if (SOA) {
            x = pts[j], y = pts[(int64_t)L.n + j], z = pts[2 * (int64_t)L.n + j];
        } else {
            const TkPoint3<T> p = tk_load3<T>(pts + (int64_t)j * 3);
            x = p.x, y = p.y, z = p.z;
        }
        const T d = tk_dist2<T>(x, y, z, cx, cy, cz);
        // The first step assigns whatever it computes (sample_farthest_points_kernel.cu:59-64
        // starts from "unset"); a NaN there never compares above anything, which -1 mimics.
        const T nm = step == 1 ? (d != d ? (T)-1 : d) : tk_min<T>(md[j], d);
        md[j] = nm;
        if (nm > (T)0 && nm >= best)
            fps_keep_better<T>(best, bpos, nm, fps_position_of_point(j, L));
    }
    fps_block_best<T, NT>(best, bpos, s_val, s_pos);
    if (tid == 0) {
        const int64_t o = ((int64_t)(step & 1) * a.batch + b) * a.groups + g;
        a.cand_val[o] = best;
        a.cand_pos[o] = bpos;
    }
}

// Workgroups per cloud and points per workgroup of the wide kernel.
inline void fps_wide_shape(int64_t B, int64_t N, int &groups, int &slice)
{
    constexpr int64_t MIN_SLICE = 2048, MAX_GROUPS = 1024;
    int64_t want = (2048 + B - 1) / B;  // about 2048 workgroups in flight
    int64_t g = (N + MIN_SLICE - 1) / MIN_SLICE;
    if (g > want)
        g = want;
    if (g > MAX_GROUPS)
        g = MAX_GROUPS;
    if (g < 1)
        g = 1;
    slice = (int)((N + g - 1) / g);
    groups = (int)((N + slice - 1) / slice);
}

template <typename T> struct FpsWideLayout {
    size_t min_dist, cand_val, cand_pos, chosen, total;
};

template <typename T> FpsWideLayout<T> fps_wide_layout(int64_t B, int64_t N, int groups)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    FpsWideLayout<T> w;
    w.min_dist = 0;
    w.cand_val = up((size_t)B * (size_t)N * sizeof(T));
    w.cand_pos = w.cand_val + up((size_t)2 * B * groups * sizeof(T));
    w.chosen = w.cand_pos + up((size_t)2 * B * groups * sizeof(int));
    w.total = w.chosen + up((size_t)2 * B * sizeof(int));
    return w;
}

FpsLayout fps_layout(int64_t n, int64_t k)
{
    FpsLayout L;
    L.n = (int)n;
    L.k = (int)k;
    int bs = 1, lg = 0;
    // Block size of the reference: smallest power of two >= n, capped at 512
    // (sample_farthest_points_kernel.cu:132-133); its switch runs 32 threads for
    // anything smaller (:153-161).
    while (bs < n && bs < 512) {
        bs *= 2;
        ++lg;
    }
    while (bs < 32) {
        bs *= 2;
        ++lg;
    }
    L.bs = bs;
    L.log2_bs = lg;
    L.c = (int)((n + bs - 1) / bs);
    L.inv_c = 1.0f / (float)L.c;
    return L;
}

// Largest number of positions the register kernel holds for element size `es`.
int64_t fps_register_capacity(size_t es) { return es == 4 ? 1024 * 16 : 1024 * 8; }

template <typename T, int P, int NT>
void fps_launch(const T *points, bool soa, int64_t B, int64_t *index, const FpsLayout &L,
                hipStream_t s)
{
    if (soa)
        hipLaunchKernelGGL((fps_register_kernel<T, P, NT, true>), dim3((unsigned)B), dim3(NT), 0,
                           s, points, index, L, 0);
    else
        hipLaunchKernelGGL((fps_register_kernel<T, P, NT, false>), dim3((unsigned)B), dim3(NT),
                           0, s, points, index, L, 0);
}

template <int P, int NT>
void fps_launch_f32(const float *points, bool soa, int64_t B, int64_t *index,
                    const FpsLayout &L, hipStream_t s)
{
    constexpr int MAXM = 6;  // 4 -> 6 gains 1-4 %, 8 nothing
    if (soa) {
        hipLaunchKernelGGL((fps_multistep_kernel_f32<P, NT, true, MAXM>), dim3((unsigned)B),
                           dim3(NT), 0, s, points, index, L);
        hipLaunchKernelGGL((fps_register_kernel<float, P, NT, true>), dim3((unsigned)B),
                           dim3(NT), 0, s, points, index, L, 1);
    } else {
        hipLaunchKernelGGL((fps_multistep_kernel_f32<P, NT, false, MAXM>), dim3((unsigned)B),
                           dim3(NT), 0, s, points, index, L);
        hipLaunchKernelGGL((fps_register_kernel<float, P, NT, false>), dim3((unsigned)B),
                           dim3(NT), 0, s, points, index, L, 1);
    }
}

// The band kernel, the check of its claims and what is left.
template <int P, int NW, int NB, bool SOA>
int fps_band_launch(const float *points, int64_t B, int64_t *index, float *sampled,
                      const FpsLayout &L, hipStream_t s)
{
    constexpr int NT = NW * TK_WAVE;
    // the sorted list, and behind it the sort's counters, then one coordinate of every point
    constexpr int LDS = NT * P * 4 + (NT * P > 4100 ? NT * P : 4100) * 4;
    constexpr auto kernel = fps_band_kernel_f32<P, NW, NB, SOA>;
    constexpr auto settle = fps_settle_kernel_f32<P, NW, NB, SOA>;
    int allowed = tk_allow_dynamic_lds<kernel>(LDS);
    if (allowed == TK3D_OK)
        allowed = tk_allow_dynamic_lds<settle>(LDS);
    if (allowed != TK3D_OK)
        return allowed;
    // up to a workgroup per 64 points: eight to a CU in all of the light first kernel, one of the second; and a
    // launch holds less than 2^32 lanes
    const auto slices = [&](int points_of, int each) {
        const int groups = (points_of + TK_WAVE - 1) / TK_WAVE;
        const int64_t most = (each * tk_cu_count() + B - 1) / B;
        return groups < most ? groups : (int)most;
    };
    const bool claims = L.k <= FPS_CLAIM_MAX && B < ((int64_t)1 << 22);
    hipLaunchKernelGGL(kernel, dim3((unsigned)B), dim3(NT), LDS, s, points, index, L, claims);
    if (claims) {
        const int of_k = slices(L.k, 8);
        hipLaunchKernelGGL((fps_claim_minima_kernel<SOA>), dim3((unsigned)(B * of_k)), dim3(1024), 0,
                           s, points, index, L, of_k);
    }
    const int of_n = slices(claims ? L.n : L.k, 1);
    hipLaunchKernelGGL(settle, dim3((unsigned)(B * of_n)), dim3(NT), LDS, s, points, index, sampled, L, of_n);
    return TK3D_OK;
}

template <int P, int NW, int NB>
int fps_band_launch_f32(const float *points, bool soa, int64_t B, int64_t *index, float *sampled,
                          const FpsLayout &L, hipStream_t s)
{
    return soa ? fps_band_launch<P, NW, NB, true>(points, B, index, sampled, L, s)
               : fps_band_launch<P, NW, NB, false>(points, B, index, sampled, L, s);
}

// fp32, the band kernel: whether it takes the call, and its launch if so. It needs 192 samples to
// be paid for: its prologue sorts the cloud, which costs 4 us at 1024 points and about 10 at 16384, and
// early in a sampling, where the points far from all centres are neighbours, a band of 64 holds one or
// two winners. Multi-step kernel against this one, with what runs behind them, us, at 128 samples (this
// one 2 to 20 us slower than now): 1 x 300 42, 35; 16 x 600 48, 55; 16 x 1024 50, 59; 16 x 4096 77, 83; 16 x 16384
// 159, 161; at 192: 65, 43; 67, 47; 69, 54; 104, 82; 222, 153. In sampling order, in which an encoder's
// levels come, it has 16 for
// 46 to 210 at 192 samples.
// Of the clouds that sixteen waves finish soonest, a CU takes two of eight waves at once, which is the faster way where
// there are more clouds than CUs. us, multi-step kernel, sixteen waves and eight: 257 x 4096 -> 192 144, 128, 94; 512 x
// 3000 -> 256 199, 165, 119; 1024 x 4096 -> 192 262, 317, 209, -> 512 602, 434, 310.
bool fps_band_dispatch_f32(const float *points, bool soa, int64_t B, int64_t *index, float *sampled,
                             const FpsLayout &L, int64_t npos, hipStream_t s, int &rc)
{
    if (npos > 1024 * 16 || L.k < 192)
        return false;
    if (npos <= 512 * 2)
        rc = fps_band_launch_f32<2, 8, 2>(points, soa, B, index, sampled, L, s);
    else if (npos <= 512 * 4)
        rc = fps_band_launch_f32<4, 8, 2>(points, soa, B, index, sampled, L, s);
    else if (npos <= 1024 * 4 && B > tk_cu_count())
        rc = fps_band_launch_f32<8, 8, 2>(points, soa, B, index, sampled, L, s);
    else if (npos <= 1024 * 4)
        rc = fps_band_launch_f32<4, 16, 2>(points, soa, B, index, sampled, L, s);
    else if (npos <= 1024 * 8)
        rc = fps_band_launch_f32<8, 16, 4>(points, soa, B, index, sampled, L, s);
    else
        rc = fps_band_launch_f32<16, 16, 4>(points, soa, B, index, sampled, L, s);
    return true;
}

// fp32, everything else that fits a workgroup: (points per lane, lanes) by cloud size, from timing
// every shape on an MI355X: two waves per SIMD (512 lanes) hide each other's reduction latency; more
// waves only repeat the per-wave reduction.
void fps_dispatch_f32(const float *points, bool soa, int64_t B, int64_t *index,
                      const FpsLayout &L, int64_t npos, hipStream_t s)
{
    if (npos <= 64 * 2)
        fps_launch_f32<2, 64>(points, soa, B, index, L, s);
    else if (npos <= 256 * 2)
        fps_launch_f32<2, 256>(points, soa, B, index, L, s);
    else if (npos <= 512 * 2)
        fps_launch_f32<2, 512>(points, soa, B, index, L, s);
    else if (npos <= 512 * 4)
        fps_launch_f32<4, 512>(points, soa, B, index, L, s);
    else if (npos <= 512 * 8)
        fps_launch_f32<8, 512>(points, soa, B, index, L, s);
    else if (npos <= 512 * 16)
        fps_launch_f32<16, 512>(points, soa, B, index, L, s);
    else
        fps_launch_f32<32, 512>(points, soa, B, index, L, s);
}

// Coordinates of the picks: sampled[b, i, :] = points[b, index[b, i], :] in the layout of
// the input cloud ([B,K,3], or [B,3,K] with SOA). A launch of its own after the
// selection kernel: storing the coordinates from the selection loop changed that loop's
// register allocation and cost it 4-9 %, far more than this pass.
template <typename T, bool SOA>
__global__ __launch_bounds__(256) void fps_gather_kernel(const T *__restrict__ points,
                                                         const int64_t *__restrict__ index,
                                                         T *__restrict__ sampled, int n, int k)
{
    const int b = blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= k)
        return;
    const T *__restrict__ pts = points + (int64_t)b * n * 3;
    T *__restrict__ so = sampled + (int64_t)b * k * 3;
    const int64_t j = index[(int64_t)b * k + i];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const T v = fps_coord<SOA>(pts, n, j, a);
        if (SOA)
            so[(int64_t)a * k + i] = v;
        else
            so[(int64_t)i * 3 + a] = v;
    }
}

template <typename T>
int fps_finish(const T *points, bool soa, int64_t B, int64_t N, int64_t K,
               const int64_t *index, T *sampled, hipStream_t s)
{
    const int rc = tk_launch_status();
    if (rc != TK3D_OK || !sampled)
        return rc;
    const dim3 grid((unsigned)((K + 255) / 256), (unsigned)B);
    if (B > 65535)
        return TK3D_ERR_UNSUPPORTED;
    if (soa)
        hipLaunchKernelGGL((fps_gather_kernel<T, true>), grid, dim3(256), 0, s, points, index,
                           sampled, (int)N, (int)K);
    else
        hipLaunchKernelGGL((fps_gather_kernel<T, false>), grid, dim3(256), 0, s, points, index,
                           sampled, (int)N, (int)K);
    return tk_launch_status();
}

template <typename T>
int fps(const T *points, bool soa, int64_t B, int64_t N, int64_t K, int64_t *index, T *sampled,
        void *workspace, size_t workspace_bytes, void *stream)
{
    if (B < 0 || N < 0)
        return TK3D_ERR_BAD_SIZE;
    if (K <= 0 || K > N)
        return TK3D_ERR_BAD_K;
    if (N > ((int64_t)1 << 23) || B > TK_MAX_I32 || !tk_fits(TK_MAX_ELEMS, B, N, 3))
        return TK3D_ERR_UNSUPPORTED;
    if (B == 0)
        return TK3D_OK;
    if (!points || !index)
        return TK3D_ERR_NULL_POINTER;
    hipStream_t s = (hipStream_t)stream;
    const FpsLayout L = fps_layout(N, K);
    const int64_t npos = (int64_t)L.bs * L.c;
    if (npos <= fps_register_capacity(sizeof(T))) {
        if constexpr (sizeof(T) == 4) {
            int rc;
            if (fps_band_dispatch_f32(points, soa, B, index, sampled, L, npos, s, rc))
                return rc != TK3D_OK ? rc : tk_launch_status();
            fps_dispatch_f32(points, soa, B, index, L, npos, s);
        } else {
            // Fewest points per lane that still covers the cloud: short serial chains.
            if (npos <= 256 * 1)
                fps_launch<T, 1, 256>(points, soa, B, index, L, s);
            else if (npos <= 256 * 2)
                fps_launch<T, 2, 256>(points, soa, B, index, L, s);
            else if (npos <= 512 * 2)
                fps_launch<T, 2, 512>(points, soa, B, index, L, s);
            else if (npos <= 1024 * 2)
                fps_launch<T, 2, 1024>(points, soa, B, index, L, s);
            else if (npos <= 1024 * 4)
                fps_launch<T, 4, 1024>(points, soa, B, index, L, s);
            else
                fps_launch<T, 8, 1024>(points, soa, B, index, L, s);
        }
        return fps_finish<T>(points, soa, B, N, K, index, sampled, s);
    }
    // Larger clouds: one launch per selection step, many workgroups per cloud.
    int groups, slice;
    fps_wide_shape(B, N, groups, slice);
    const FpsWideLayout<T> w = fps_wide_layout<T>(B, N, groups);
    if (!workspace || workspace_bytes < w.total || ((uintptr_t)workspace & 7) != 0)
        return TK3D_ERR_WORKSPACE;
    if (B > 65535)
        return TK3D_ERR_UNSUPPORTED;
    char *base = (char *)workspace;
    FpsWideArgs<T> a;
    a.points = points;
    a.index = index;
    a.min_dist = (T *)(base + w.min_dist);
    a.cand_val = (T *)(base + w.cand_val);
    a.cand_pos = (int *)(base + w.cand_pos);
    a.chosen = (int *)(base + w.chosen);
    a.groups = groups;
    a.slice = slice;
    a.batch = (int)B;
    const dim3 grid((unsigned)groups, (unsigned)B);
    for (int64_t step = 1; step <= K; ++step) {
        // The last launch has nothing to update: one workgroup per cloud records the choice.
        const dim3 gr = step == K ? dim3(1u, (unsigned)B) : grid;
        if (soa)
            hipLaunchKernelGGL((fps_wide_step_kernel<T, 256, true>), gr, dim3(256), 0, s, a, L,
                               (int)step);
        else
            hipLaunchKernelGGL((fps_wide_step_kernel<T, 256, false>), gr, dim3(256), 0, s, a, L,
                               (int)step);
    }
    return fps_finish<T>(points, soa, B, N, K, index, sampled, s);
}

// Workspace of tk3d_sample_farthest_points_static_f32: lives in the library's device
// image, one copy per GPU, for callers that cannot allocate. In host code the array's
// name is only a handle for hipGetSymbolAddress; kernels are handed the address that
// call returns for the current device.
__device__ __align__(256) unsigned char fps_static_scratch[TK3D_FPS_STATIC_WORKSPACE_BYTES];

// Device address of fps_static_scratch on the current device, looked up once per device.
int fps_static_scratch_address(void **address)
{
    constexpr int MAX_DEVICES = 64;
    static std::atomic<void *> known[MAX_DEVICES];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES)
        return TK3D_ERR_UNSUPPORTED;
    void *p = known[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(fps_static_scratch));
        if (e != hipSuccess)
            return (int)e;
        if (!p)
            return TK3D_ERR_WORKSPACE;
        known[dev].store(p, std::memory_order_release);  // every thread finds the same value
    }
    *address = p;
    return TK3D_OK;
}

}  // namespace

extern "C" {

size_t tk3d_sample_farthest_points_workspace_bytes(int64_t B, int64_t N, size_t elem_size)
{
    if (B <= 0 || N <= 0 || (elem_size != 4 && elem_size != 8))
        return 0;
    const FpsLayout L = fps_layout(N, 1);
    const int64_t npos = (int64_t)L.bs * L.c;
    if (npos <= fps_register_capacity(elem_size))
        return 0;
    int groups, slice;
    fps_wide_shape(B, N, groups, slice);
    return elem_size == 4 ? fps_wide_layout<float>(B, N, groups).total
                          : fps_wide_layout<double>(B, N, groups).total;
}

int tk3d_sample_farthest_points_f32(const float *points, int64_t B, int64_t N,
                                    int64_t num_samples, int64_t *index, void *workspace,
                                    size_t workspace_bytes, void *stream)
{
    return fps<float>(points, false, B, N, num_samples, index, nullptr, workspace,
                      workspace_bytes, stream);
}

int tk3d_sample_farthest_points_static_f32(const float *points, int64_t B, int64_t N,
                                           int64_t num_samples, int64_t *index, void *stream)
{
    const size_t need = tk3d_sample_farthest_points_workspace_bytes(B, N, sizeof(float));
    if (need > (size_t)TK3D_FPS_STATIC_WORKSPACE_BYTES)
        return TK3D_ERR_WORKSPACE;
    void *scratch = nullptr;
    if (need > 0) {
        const int rc = fps_static_scratch_address(&scratch);
        if (rc != TK3D_OK)
            return rc;
    }
    // Nothing in the workspace has to start at zero: the first step assigns every running
    // minimum and each later step reads only what the step before it wrote.
    return fps<float>(points, false, B, N, num_samples, index, nullptr, scratch,
                      need > 0 ? (size_t)TK3D_FPS_STATIC_WORKSPACE_BYTES : 0, stream);
}

int tk3d_sample_farthest_points_f64(const double *points, int64_t B, int64_t N,
                                    int64_t num_samples, int64_t *index, void *workspace,
                                    size_t workspace_bytes, void *stream)
{
    return fps<double>(points, false, B, N, num_samples, index, nullptr, workspace,
                       workspace_bytes, stream);
}

int tk3d_sample_farthest_points_gather_f32(const float *points, int channels_first,
                                           int64_t B, int64_t N, int64_t num_samples,
                                           int64_t *index, float *sampled, void *workspace,
                                           size_t workspace_bytes, void *stream)
{
    return fps<float>(points, channels_first != 0, B, N, num_samples, index, sampled,
                      workspace, workspace_bytes, stream);
}

int tk3d_sample_farthest_points_gather_f64(const double *points, int channels_first,
                                           int64_t B, int64_t N, int64_t num_samples,
                                           int64_t *index, double *sampled, void *workspace,
                                           size_t workspace_bytes, void *stream)
{
    return fps<double>(points, channels_first != 0, B, N, num_samples, index, sampled,
                       workspace, workspace_bytes, stream);
}

}  // extern "C"
