// fss_direct.hip -- O(N^2) direct sum (rhs_direct_sum, Old-BVE-code/rhs_eval.h:15-32,
// followed by the rhs_func scaling, rhs_eval.h:54-55).
//
// Work is cut into (group of 64 R targets, wave tile of sources) units: a lane
// holds R targets, a wave stages one tile at a time in its own LDS slice and
// the block's four waves take the tiles of a segment in turn, so nothing in
// the source loop waits for another wave.  Below DIRECT_SPLIT_GROUPS target
// groups the units, flattened group by group, are cut into runs of equal
// length (direct_plan; a run may end inside a group), a block per run; every
// block leaves one partial per group it touched and k_direct_sum adds them in a
// fixed order.  Beyond that a block takes a whole group and writes the
// velocities itself.
//
// FP64 sums of all particles are taken over unordered pairs from 3,300
// particles on (k_direct_sym); these kernels do smaller ones, chosen targets and
// mixed precision.
//
// Bound by FP64 issue (17 four-cycle slots a pair at four targets a lane: 10,000
// targets of N = 655,362 in 3.4 ms, 1.95e12 pairs/s at about 2 GHz).  One target a
// lane, one block per 256 targets and a reciprocal with two Newton steps per pair
// took 42.6 ms there, and for the full sums that k_direct_sym now takes 2,036 us
// at N = 40,009 (these kernels 822) and 525 us at N = 10,242 (79).
//
// The self pair j == i is skipped as the reference does (rhs_eval.h:20); only
// tiles that hold a target of the wave pay for the index test.
//
// FP64: reference kernel (x_i x x_j) w_j / (1 - x_i . x_j) with the
//       reference's unfused x.y, factored as
//       x_i x sum_j (w_j / (1 - x_i.x_j)) (x_j - x_i)  (no cancellation for
//       near pairs); one reciprocal for the R denominators of a lane.
// FP32 (mixed): 1 - x.y = |x - y|^2 / 2 on the sphere, d = x_j - x_i,
//       x_i x x_j = x_i x d; per-tile FP32 partial sums are added into FP64
//       accumulators (256 terms per partial), the cross product and scaling
//       are FP64.
#include <algorithm>
#include <cmath>
#include <functional>
#include <initializer_list>
#include <mutex>

#include "fss_internal.h"
#include "fss_rk4_dev.h"

namespace fss {

__device__ inline double rcp64d(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    double e = fma(-d, r, 1.0);
    r = fma(r, e, r);
    e = fma(-d, r, 1.0);
    r = fma(r, e, r);
    return r;
}

__global__ void k_pack64(const double *__restrict__ x, const double *__restrict__ y,
                         const double *__restrict__ z, const double *__restrict__ vort,
                         const double *__restrict__ area, int64_t n, double4 *src, uint64_t *ts)
{
    stamp_start(ts, Timing::START);
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) src[i] = make_double4(x[i], y[i], z[i], vort[i] * area[i]);
}

__global__ void k_pack32(const double *__restrict__ x, const double *__restrict__ y,
                         const double *__restrict__ z, const double *__restrict__ vort,
                         const double *__restrict__ area, int64_t n, float4 *src, uint64_t *ts)
{
    stamp_start(ts, Timing::START);
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) src[i] = make_float4((float)x[i], (float)y[i], (float)z[i], 2.0f * (float)(vort[i] * area[i]));
}

// Target groups of 256 from which a block takes a whole group (10 a CU: the
// last blocks then idle at most a tenth of the chip); below it the partials fit
// FSS_DIRECT_SCRATCH_BYTES.
constexpr int64_t DIRECT_SPLIT_GROUPS = 2560;

template <typename Real> struct Dir;
template <> struct Dir<double> {
    using T4 = double4;
};
template <> struct Dir<float> {
    using T4 = float4;
};

struct DirectArgs {
    const double *x, *y, *z, *vort, *area;
    const void *rec; // packed records (whole groups only)
    const int64_t *idx;
    int64_t n, m;
    int64_t K, U;     // wave tiles per group, units
    int64_t B1, q1, q; // units of block b: q1 for b < B1, then q
    double scale, omega;
    double *part;
    double *u, *v, *w, *dvort;
    uint64_t *ts; // time stamps, or null
};

template <typename Args> __device__ inline void direct_source(const Args &a, int64_t j, double4 &s)
{
    s = make_double4(a.x[j], a.y[j], a.z[j], a.vort[j] * a.area[j]);
}
// FP32 sources carry the doubled weight: 2 w / |d|^2 = w / (|d|^2 / 2), the
// same bits (a factor of two is exact) with one multiplication less per pair
__device__ inline void direct_source(const DirectArgs &a, int64_t j, float4 &s)
{
    s = make_float4((float)a.x[j], (float)a.y[j], (float)a.z[j], 2.0f * (float)(a.vort[j] * a.area[j]));
}

// One FP64 source against the R targets of a lane: prefix products P_q =
// den_0 ... den_q, r = w / P_{R-1}, then backward c_q = P_{q-1} r, r <- den_q r:
// one v_rcp_f64 (quarter rate) and two Newton steps for R pairs instead of for
// each.  A product that is zero, infinite or not a number in any lane (a pair
// of coincident points; positions far off the sphere) takes the wave through
// one reciprocal per pair.
template <int R, bool MASK>
__device__ inline void direct_eval(const double4 *xt, const double4 &s, int k, const int *self, double (*S)[3])
{
    double den[R], pre[R], c[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
        double dot;
        {
            // x.y summed as the reference does (helpers.h:23-28): no FMA
#pragma clang fp contract(off)
            dot = xt[q].x * s.x;
            dot = dot + xt[q].y * s.y;
            dot = dot + xt[q].z * s.z;
        }
        den[q] = 1.0 - dot;
        if (MASK) den[q] = k == self[q] ? 1.0 : den[q];
        pre[q] = q == 0 ? den[0] : pre[q - 1] * den[q];
    }
    if (R == 1 || __builtin_amdgcn_ballot_w64(!__builtin_amdgcn_class(pre[R - 1], 0x108)) == 0) { // normal numbers
        double rw = s.w * rcp64d(pre[R - 1]);
#pragma unroll
        for (int q = R - 1; q > 0; q--) {
            c[q] = pre[q - 1] * rw;
            rw = den[q] * rw;
        }
        c[0] = rw;
    } else {
#pragma unroll
        for (int q = 0; q < R; q++) c[q] = s.w * rcp64d(den[q]);
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        if (MASK) c[q] = k == self[q] ? 0.0 : c[q];
        S[q][0] = fma(c[q], s.x - xt[q].x, S[q][0]);
        S[q][1] = fma(c[q], s.y - xt[q].y, S[q][1]);
        S[q][2] = fma(c[q], s.z - xt[q].z, S[q][2]);
    }
}
template <int R, bool MASK>
__device__ inline void direct_eval(const float4 *xt, const float4 &s, int k, const int *self, float (*S)[3])
{
#pragma unroll
    for (int q = 0; q < R; q++) {
        float dx = s.x - xt[q].x, dy = s.y - xt[q].y, dz = s.z - xt[q].z;
        float den = dx * dx + dy * dy + dz * dz;
        float c = s.w * __builtin_amdgcn_rcpf(den);
        if (MASK) c = k == self[q] ? 0.0f : c;
        S[q][0] = fmaf(c, dx, S[q][0]);
        S[q][1] = fmaf(c, dy, S[q][1]);
        S[q][2] = fmaf(c, dz, S[q][2]);
    }
}

// a tile's sums into the FP64 accumulators
template <int R, bool MASK>
__device__ inline void direct_tile(const double4 *xt, const double4 *tile, int cnt, const int *self, double (*S)[3])
{
    constexpr int UN = R == 1 ? 4 : 1; // the loop with a wave-wide test is not unrolled
#pragma unroll UN
    for (int k = 0; k < cnt; k++) direct_eval<R, MASK>(xt, tile[k], k, self, S);
}
template <int R, bool MASK>
__device__ inline void direct_tile(const float4 *xt, const float4 *tile, int cnt, const int *self, double (*S)[3])
{
    constexpr int UN = 8 / R;
    float P[R][3] = {};
#pragma unroll UN
    for (int k = 0; k < cnt; k++) direct_eval<R, MASK>(xt, tile[k], k, self, P);
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
        for (int c = 0; c < 3; c++) S[q][c] += (double)P[q][c];
}

__device__ inline void direct_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// first unit of block b, and the block of unit u
__host__ __device__ inline int64_t direct_first(int64_t b, int64_t B1, int64_t q1, int64_t q)
{
    return b < B1 ? b * q1 : B1 * q1 + (b - B1) * q;
}
__device__ inline int64_t direct_block(int64_t u, int64_t B1, int64_t q1, int64_t q)
{
    return u < B1 * q1 ? u / q1 : B1 + (u - B1 * q1) / q;
}

template <typename Real, int R, int WT, bool SPLIT>
__global__ void __launch_bounds__(256, 4) k_direct(DirectArgs a)
{
    using T4 = typename Dir<Real>::T4;
    constexpr int SL = (WT + 63) / 64, NT = 64 * R;
    constexpr int TILE_BYTES = (int)sizeof(T4) * WT * 4, RED_BYTES = 8 * 4 * NT;
    __shared__ __align__(32) unsigned char smem[TILE_BYTES > RED_BYTES ? TILE_BYTES : RED_BYTES];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    T4 *tile = reinterpret_cast<T4 *>(smem) + wave * WT;
    double *red = reinterpret_cast<double *>(smem); // [4][NT], after a segment's last tile
    const T4 *rec = static_cast<const T4 *>(a.rec);
    if (SPLIT) stamp_start(a.ts, Timing::START);
    stamp_start(a.ts, Timing::MAIN);
    const int64_t b = blockIdx.x;
    int64_t u = direct_first(b, a.B1, a.q1, a.q);
    const int64_t u1 = min(u + (b < a.B1 ? a.q1 : a.q), a.U);
    while (u < u1) {
        const int64_t g = u / a.K, t0 = u - g * a.K, t1 = min(a.K, t0 + (u1 - u));
        T4 xt[R];
        double S[R][3];
        auto target = [&](int q) {
            const int64_t r = min(g * NT + 64 * q + lane, a.m - 1);
            return a.idx ? a.idx[r] : r;
        };
        int64_t id[R];
#pragma unroll
        for (int q = 0; q < R; q++) {
            id[q] = target(q);
            if (SPLIT) direct_source(a, id[q], xt[q]);
            else xt[q] = rec[id[q]];
            S[q][0] = S[q][1] = S[q][2] = 0.0;
        }
        T4 nx[SL];
        auto fetch = [&](int64_t t) {
#pragma unroll
            for (int s = 0; s < SL; s++) {
                const int64_t j = min(t * WT + 64 * s + (WT < 64 ? lane % WT : lane), a.n - 1);
                if (SPLIT) direct_source(a, j, nx[s]);
                else nx[s] = rec[j];
            }
        };
        int64_t t = t0 + wave;
        if (t < t1) fetch(t);
        for (; t < t1; t += 4) {
#pragma unroll
            for (int s = 0; s < SL; s++)
                if (WT >= 64 || lane < WT) tile[64 * s + lane] = nx[s];
            direct_wave_sync();
            if (t + 4 < t1) fetch(t + 4);
            const int64_t base = t * WT;
            const int cnt = (int)min((int64_t)WT, a.n - base);
            int self[R];
            bool any = false;
            // four targets are read again for each tile: kept, they would cost
            // eight registers
            if (a.idx || (base < (g + 1) * NT && base + WT > g * NT)) {
#pragma unroll
                for (int q = 0; q < R; q++) {
                    const int64_t o = (R < 4 ? id[q] : target(q)) - base;
                    self[q] = o >= 0 && o < WT ? (int)o : -1;
                    any = any || self[q] >= 0;
                }
            }
            if (__any(any)) direct_tile<R, true>(xt, tile, cnt, self, S);
            else direct_tile<R, false>(xt, tile, cnt, self, S);
            direct_wave_sync();
        }
        // sum over the four waves in order, one component at a time (4 NT
        // doubles of LDS); thread o < NT then holds target o of the group
        double sum[3];
        const int o = threadIdx.x;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < R; q++) red[wave * NT + 64 * q + lane] = S[q][c];
            __syncthreads();
            if (o < NT) sum[c] = ((red[o] + red[NT + o]) + red[2 * NT + o]) + red[3 * NT + o];
        }
        __syncthreads();
        const int64_t r = g * NT + o;
        if (o < NT && r < a.m) {
            const int64_t i = a.idx ? a.idx[r] : r;
            T4 xi;
            if (SPLIT) direct_source(a, i, xi);
            else xi = rec[i];
            const double x0 = xi.x, x1 = xi.y, x2 = xi.z;
            const double a0 = (x1 * sum[2] - x2 * sum[1]) * a.scale;
            const double a1 = (x2 * sum[0] - x0 * sum[2]) * a.scale;
            const double a2 = (x0 * sum[1] - x1 * sum[0]) * a.scale;
            if (SPLIT) {
                // the partials of a run of units have the distinct numbers
                // block + group: every step of the run raises one of them
                double *pt = a.part + ((int64_t)blockIdx.x + g) * 3 * NT + o;
                pt[0] = a0;
                pt[NT] = a1;
                pt[2 * NT] = a2;
            } else {
                a.u[r] = a0;
                a.v[r] = a1;
                a.w[r] = a2;
                a.dvort[r] = -2 * a.omega * a2;
            }
        }
        u += t1 - t0;
    }
    if (!SPLIT) stamp_end(a.ts);
}

// sums the partials of every target over the blocks of its group: 16 targets x
// 16 ways per block (a few thousand targets have up to 50 partials each, and
// one thread per target would walk them alone), ways added in order
__global__ void __launch_bounds__(256) k_direct_sum(const double *__restrict__ part, int64_t m, int nt, int64_t K,
                                                    int64_t B1, int64_t q1, int64_t q, double omega, double *u, double *v, double *w,
                                                    double *dvort, RkNext next, uint64_t *ts)
{
    __shared__ double red[3][16][17];
    const int tl = threadIdx.x & 15, way = threadIdx.x >> 4;
    const int64_t r = min((int64_t)blockIdx.x * 16 + tl, m - 1), g = r / nt;
    const int64_t b0 = direct_block(g * K, B1, q1, q), b1 = direct_block((g + 1) * K - 1, B1, q1, q);
    double s[3] = {0, 0, 0};
#pragma unroll 4
    for (int64_t b = b0 + way; b <= b1; b += 16) {
        const double *pt = part + (b + g) * 3 * nt + (r - g * nt);
        s[0] += pt[0];
        s[1] += pt[nt];
        s[2] += pt[2 * nt];
    }
    for (int c = 0; c < 3; c++) red[c][way][tl] = s[c];
    __syncthreads();
    if (way < 3) {
        double t = 0;
        for (int h = 0; h < 16; h++) t += red[way][h][tl];
        red[way][0][tl] = t;
    }
    __syncthreads();
    if (way == 0 && (int64_t)blockIdx.x * 16 + tl < m) {
        const double a0 = red[0][0][tl], a1 = red[1][0][tl], a2 = red[2][0][tl], a3 = -2 * omega * a2;
        if (next.mode != RkNext::STEP) {
            u[r] = a0;
            v[r] = a1;
            w[r] = a2;
            dvort[r] = a3;
        }
        rk_next(next, r, a0, a1, a2, a3);
    }
    stamp_end(ts);
}

// ------------------------------------------------------------------
// FP64 sum over unordered pairs: 1 - x.y and its reciprocal serve both
// directions of a pair
// ------------------------------------------------------------------
// k_direct runs at the FP64 issue rate, so only fewer instructions help: a pair
// in both directions takes 21.5 four-cycle slots at four targets a lane against
// 2 x 17.  A block holds a row of T = 256 R targets (R a lane, w_i with them) and
// walks the tiles of 64 particles from the row's own on.  In a tile every lane
// starts at its own source and takes the next lane's at each of 64 steps (read
// from LDS), while the sums of the sources travel the ring of lanes the other
// way by one DPP move a word (a tenth of a step); after 64 steps every source's
// sum is back with its lane, the four waves' are added and stored as column sums
// of the row.  The row's own tiles take their pairs in one direction, which
// keeps the self test and the remainders out of the main loop.  k_sym_sum adds
// each target's column and run sums in a fixed order; rows go in slabs so that
// both fit a bounded workspace.  N = 100,003: 1.98e12 -> 2.56e12 ordered pairs/s
// (102 cycles a step and target at about 2 GHz, 98 of them issue).
struct SymArgs {
    const double *x, *y, *z, *vort, *area;
    int64_t n, K;      // particles, tiles of 64 of them
    int64_t r0, r1;    // rows of targets of this launch
    int64_t U, B1, q1, q; // its units, and their cut into runs
    double scale, omega;
    double *col, *part;
    double *u, *v, *w, *dvort;
    uint64_t *ts;
};

// Row r: targets [r T, (r + 1) T); its units are the tiles r RT .. K - 1 (RT = T /
// 64), numbered row by row from row r0; its column sums are those of the
// particles after the row.
__host__ __device__ inline int64_t sym_first(int64_t r, int64_t r0, int64_t K, int64_t RT)
{
    return (r - r0) * K - RT * (r * (r - 1) - r0 * (r0 - 1)) / 2;
}
__host__ __device__ inline int64_t sym_cols(int64_t r, int64_t K, int64_t T)
{
    return 64 * K > (r + 1) * T ? 64 * K - (r + 1) * T : 0;
}
__host__ __device__ inline int64_t sym_col_first(int64_t r, int64_t r0, int64_t K, int64_t T)
{
    return (r - r0) * 64 * K - T * (r * (r + 1) - r0 * (r0 + 1)) / 2;
}

// the value of a neighbouring lane, the wave taken as a ring
__device__ inline int ring(int v) { return __builtin_amdgcn_mov_dpp(v, 0x134, 0xf, 0xf, false); }
__device__ inline double ring(double v)
{
    return __hiloint2double(ring(__double2hiint(v)), ring(__double2loint(v)));
}

// One FP64 source of the lane against its R targets, both directions: c_q = w_j
// / den_q goes to the targets' sums S, w_q / den_q to the source's A (with the
// sign of x_j - x_q; the caller turns it).
template <int R>
__device__ inline void sym_eval(const double4 *xt, const double4 &s, double (*S)[3], double *A)
{
    double d[R][3], den[R], pre[R], c[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
        double dot;
        {
#pragma clang fp contract(off)
            dot = xt[q].x * s.x;
            dot = dot + xt[q].y * s.y;
            dot = dot + xt[q].z * s.z;
        }
        den[q] = 1.0 - dot;
        pre[q] = q == 0 ? den[0] : pre[q - 1] * den[q];
        d[q][0] = s.x - xt[q].x;
        d[q][1] = s.y - xt[q].y;
        d[q][2] = s.z - xt[q].z;
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!__builtin_amdgcn_class(pre[R - 1], 0x108)) == 0, 1)) { // normal numbers
        double r = rcp64d(pre[R - 1]);
#pragma unroll
        for (int q = R - 1; q > 0; q--) {
            c[q] = pre[q - 1] * r;
            r = den[q] * r;
        }
        c[0] = r;
    } else {
#pragma unroll
        for (int q = 0; q < R; q++) c[q] = rcp64d(den[q]);
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        const double cs = c[q] * s.w, ct = c[q] * xt[q].w;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            S[q][k] = fma(cs, d[q][k], S[q][k]);
            A[k] = fma(ct, d[q][k], A[k]);
        }
    }
}

template <int R>
__global__ void __launch_bounds__(256, R == 4 ? 3 : 4) k_direct_sym(SymArgs a)
{
    constexpr int T = 256 * R, RT = 4 * R;
    __shared__ __align__(16) double2 txy[2][64], tzw[2][64]; // tiles in turn: (x, y), (z, w)
    __shared__ double red[2][4][3][64];                       // a tile's column sums of the four waves
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    stamp_start(a.ts, Timing::START);
    stamp_start(a.ts, Timing::MAIN);
    const int64_t b = blockIdx.x;
    int64_t u = direct_first(b, a.B1, a.q1, a.q);
    const int64_t u1 = min(u + (b < a.B1 ? a.q1 : a.q), a.U);
    int64_t row = a.r0;
    // thread (component, source) of the tile that is fetched
    auto fetch = [&](int64_t t) {
        const int64_t j = min(64 * t + lane, a.n - 1);
        return wave == 0 ? a.x[j] : wave == 1 ? a.y[j] : wave == 2 ? a.z[j] : 64 * t + lane < a.n ? a.vort[j] * a.area[j] : 0.0;
    };
    while (u < u1) {
        while (sym_first(row + 1, a.r0, a.K, RT) <= u) row++;
        const int64_t t0 = row * RT + u - sym_first(row, a.r0, a.K, RT), t1 = min(a.K, t0 + (u1 - u));
        double4 xt[R];
        double S[R][3];
#pragma unroll
        for (int q = 0; q < R; q++) {
            direct_source(a, min(row * T + 64 * (wave * R + q) + lane, a.n - 1), xt[q]);
            S[q][0] = S[q][1] = S[q][2] = 0.0;
        }
        double *col = a.col + 3 * sym_col_first(row, a.r0, a.K, T) - (row + 1) * T;
        const int64_t len = sym_cols(row, a.K, T);
        // column sums of tile t, left in red[i] by the four waves
        auto store = [&](int i, int64_t t) {
            if (wave < 3) {
                const double v = ((red[i][0][wave][lane] + red[i][1][wave][lane]) + red[i][2][wave][lane]) + red[i][3][wave][lane];
                col[wave * len + 64 * t + lane] = -v;
            }
        };
        double nx = fetch(t0);
        int i = 0;
        for (int64_t t = t0; t < t1; t++, i ^= 1) {
            reinterpret_cast<double *>(wave < 2 ? &txy[i][lane] : &tzw[i][lane])[wave & 1] = nx;
            // one barrier a tile: it ends the stores to this tile's buffer and
            // the reads of the other one, both of two tiles ago and of the last
            __syncthreads();
            if (t > t0 && t - 1 >= (row + 1) * RT) store(i ^ 1, t - 1);
            if (t + 1 < t1) nx = fetch(t + 1);
            if (t >= (row + 1) * RT) {
                double A[3] = {0, 0, 0};
                int at = lane;
                double2 p = txy[i][at], zw = tzw[i][at];
#pragma unroll 2
                for (int k = 0; k < 64; k++) {
                    const double4 s = make_double4(p.x, p.y, zw.x, zw.y);
                    at = ring(at);
                    p = txy[i][at];
                    zw = tzw[i][at];
                    sym_eval<R>(xt, s, S, A);
#pragma unroll
                    for (int c = 0; c < 3; c++) A[c] = ring(A[c]);
                }
#pragma unroll
                for (int c = 0; c < 3; c++) red[i][wave][c][lane] = A[c];
            } else {
                // a tile of the row itself: its pairs in one direction
                const int cnt = (int)min((int64_t)64, a.n - 64 * t);
                int self[R];
#pragma unroll
                for (int q = 0; q < R; q++) self[q] = t == row * RT + wave * R + q ? lane : -1;
                for (int k = 0; k < cnt; k++)
                    direct_eval<R, true>(xt, make_double4(txy[i][k].x, txy[i][k].y, tzw[i][k].x, tzw[i][k].y), k, self, S);
            }
        }
        __syncthreads();
        if (t1 - 1 >= (row + 1) * RT) store(i ^ 1, t1 - 1);
        double *pt = a.part + (b + (row - a.r0)) * 3 * T + wave * 64 * R + lane;
#pragma unroll
        for (int q = 0; q < R; q++)
#pragma unroll
            for (int c = 0; c < 3; c++) pt[c * T + 64 * q] = S[q][c];
        u += t1 - t0;
    }
}

// adds a slab's column and run sums of every target from its first row on, 16
// targets x 16 ways per block, ways added in order; the velocities of a
// target are written by the first slab and raised by the others
template <int R> __global__ void __launch_bounds__(256) k_sym_sum(SymArgs a, RkNext next)
{
    constexpr int T = 256 * R, RT = 4 * R;
    __shared__ double red[3][16][17];
    const int tl = threadIdx.x & 15, way = threadIdx.x >> 4;
    const int64_t at = a.r0 * T + (int64_t)blockIdx.x * 16 + tl, j = min(at, a.n - 1), row = j / T;
    double s[3] = {0, 0, 0};
#pragma unroll 4
    for (int64_t r = a.r0 + way; r < min(row, a.r1); r += 16) {
        const int64_t len = sym_cols(r, a.K, T);
        const double *c = a.col + 3 * sym_col_first(r, a.r0, a.K, T) + (j - (r + 1) * T);
        s[0] += c[0];
        s[1] += c[len];
        s[2] += c[2 * len];
    }
    if (row < a.r1) {
        const int64_t b0 = direct_block(sym_first(row, a.r0, a.K, RT), a.B1, a.q1, a.q);
        const int64_t b1 = direct_block(sym_first(row + 1, a.r0, a.K, RT) - 1, a.B1, a.q1, a.q);
#pragma unroll 4
        for (int64_t b = b0 + way; b <= b1; b += 16) {
            const double *pt = a.part + (b + (row - a.r0)) * 3 * T + (j - row * T);
            s[0] += pt[0];
            s[1] += pt[T];
            s[2] += pt[2 * T];
        }
    }
    for (int c = 0; c < 3; c++) red[c][way][tl] = s[c];
    __syncthreads();
    if (way < 3) {
        double t = 0;
        for (int h = 0; h < 16; h++) t += red[way][h][tl];
        red[way][0][tl] = t;
    }
    __syncthreads();
    if (way == 0 && at < a.n) {
        const double x0 = a.x[j], x1 = a.y[j], x2 = a.z[j];
        const double s0 = red[0][0][tl], s1 = red[1][0][tl], s2 = red[2][0][tl];
        double v0 = (x1 * s2 - x2 * s1) * a.scale, v1 = (x2 * s0 - x0 * s2) * a.scale, v2 = (x0 * s1 - x1 * s0) * a.scale;
        if (a.r0 > 0) {
            v0 += a.u[j];
            v1 += a.v[j];
            v2 += a.w[j];
        }
        const double v3 = -2 * a.omega * v2;
        // a target is done with its own row's slab, and later slabs read neither
        // it nor its state
        const bool done = row < a.r1;
        if (!done || next.mode != RkNext::STEP) {
            a.u[j] = v0;
            a.v[j] = v1;
            a.w[j] = v2;
            a.dvort[j] = v3;
        }
        if (done) rk_next(next, j, v0, v1, v2, v3);
    }
    stamp_end(a.ts);
}

struct DirectPlan {
    int R, wt; // targets per lane, sources per wave tile
    bool split;
    int64_t K, G, U, B1, q1, q, B;
};

// Layout of a call.  A lane's targets share a reciprocal and each LDS read, but
// a wave then runs longer on its own (the lone-wave time of a tile) and fewer
// waves exist, so few pairs take few targets a lane: the layout with the least
//   lone-wave time + padded pairs / rate,
// both measured (us, pairs per us).  FP64, N = 2,562 / 10,242 / 40,009: one
// target and 16-source tiles 12.7 / 97 / 1,130 us, one and 64-source tiles 19 /
// 88 / 983, two 22 / 79 / 893, four 33 / 84 / 822.  FP32, whose tile of 256 sources is one FP32 partial sum: one
// target 20 / 46 / 417 us, two 34 / 54 / 399, four 63 / 78 / 425 (never the
// best).
struct DirectLayout {
    int R, wt;
    double lone, rate;
};
static const DirectLayout kDirect64[4] = {
    {1, 16, 4, 0.9e6}, {1, 64, 15, 1.5e6}, {2, 64, 20, 1.84e6}, {4, 64, 27, 1.95e6}};
static const DirectLayout kDirect32[2] = {{1, 256, 20, 4.0e6}, {2, 256, 34, 4.4e6}};
struct Layouts {
    const DirectLayout *first, *last;
    const DirectLayout *begin() const { return first; }
    const DirectLayout *end() const { return last; }
};
static Layouts direct_layouts(bool mixed) { return mixed ? Layouts{kDirect32, kDirect32 + 2} : Layouts{kDirect64, kDirect64 + 4}; }

static DirectPlan direct_plan(int64_t n, int64_t m, bool mixed)
{
    DirectPlan p{};
    const Layouts lay = direct_layouts(mixed);
    p.split = div_up(m, 256) < DIRECT_SPLIT_GROUPS;
    const DirectLayout *pick = lay.last - 1;
    double best = INFINITY;
    for (const DirectLayout *l = lay.first; l < lay.last && p.split; l++) {
        const double t = l->lone + (double)(div_up(m, 64 * l->R) * 64 * l->R) * (double)n / l->rate;
        if (t < best) {
            best = t;
            pick = l;
        }
    }
    p.R = pick->R;
    p.wt = pick->wt;
    p.K = div_up(n, p.wt);
    p.G = div_up(m, 64 * p.R);
    p.U = p.G * p.K;
    if (!p.split) {
        p.q = p.K;
        p.B = p.G;
        return p;
    }
    // Runs, in quads of units (one per wave): up to about two rounds of the
    // 1,024 resident blocks one quad each; above, three quarters of the work in
    // one round of long runs and the rest in short ones, so that the blocks that
    // end last are short (equal runs in two rounds: 872 us at N = 40,009, in
    // four 841).  A group of fewer than four tiles is a run of its own: in a quad
    // with the next group's tiles it would wait for them (mixed, N = 257: a call of
    // 24 us, now 15).  The partials of all of them stay within 30 MiB.
    const int64_t V = div_up(p.U, 4), slots = 1024;
    const int64_t most = ((int64_t)30 << 20) / (1536 * p.R) - p.G; // no fewer than the groups
    if (p.K < 4) {
        p.q = p.K;
    } else if (V <= std::min<int64_t>(2 * slots, most)) {
        p.q = 4;
    } else {
        p.B1 = slots;
        p.q1 = 4 * (3 * V / (4 * slots));
        const int64_t rest = V - p.B1 * (p.q1 / 4);
        p.q = 4 * div_up(rest, std::min<int64_t>(3 * slots, most - slots));
    }
    p.B = p.B1 + div_up(std::max<int64_t>(0, p.U - p.B1 * p.q1), p.q);
    return p;
}

// Bytes of workspace that serve every plan of n particles and m targets or fewer of
// either, in whatever layout: a call may be captured after an eager one that was no
// smaller, and must not allocate then.  Partials: a run has at least four units or
// a group's, and a plan at most 4,096 runs or one per group.
static size_t direct_bytes(int64_t n, int64_t m, bool mixed)
{
    const bool whole = div_up(m, 256) >= DIRECT_SPLIT_GROUPS;
    int64_t bytes = whole ? (mixed ? sizeof(float4) : sizeof(double4)) * n : 0;
    const int64_t ms = std::min<int64_t>(m, 256 * (DIRECT_SPLIT_GROUPS - 1));
    for (const DirectLayout &l : direct_layouts(mixed)) {
        const int64_t G = div_up(ms, 64 * l.R), V = div_up(G * div_up(n, l.wt), 4);
        bytes = std::max(bytes, std::min((int64_t)30 << 20, 1536 * l.R * (std::max(G, std::min<int64_t>(V, 4096)) + G)));
    }
    return (size_t)bytes;
}

// Workspace of the sum over unordered pairs, within the allocation-free variant's
// scratch.  With 30 MiB 20,011 particles have room for equal runs only (187 us,
// now 165) and 100,003 take 10 slabs (3,904 us, now 3 and 3,730); 126 MiB gave 0.5
// to 4 % more.
constexpr int64_t DIRECT_SCRATCH = (int64_t)64 << 20, SYM_BYTES = (int64_t)62 << 20;
static_assert(DIRECT_SCRATCH >= (int64_t)FSS_DIRECT_SCRATCH_BYTES, "records of the largest sum");

// Targets per lane of the sum over unordered pairs, or 0 where k_direct does
// the call: chosen targets and mixed precision (whose FP32 partial sums keep
// their order), few particles, whose units are fewer than the resident blocks,
// and more than one row's column sums have room for.  Us a call, k_direct
// against two / four targets a lane: N = 2,562 14.3, 17.3 / 22.1; 3,500 21.7, 18.6 /
// 23.6; 10,242 75.3, 59.8 / 60.5; 15,000 146.7, 105.9 / 116.7; 20,011 233.4, 197.1 /
// 186.3; 40,009 824, 705 / 630; 100,003 5,045, 4,361 / 3,902 (with 30 MiB); 655,362
// 228,600, - / 159,600.
static int sym_targets(int64_t n, const int64_t *idx, bool mixed)
{
    if (idx || mixed || n < 3300 || n > 1900000) return 0;
    return n < 18000 ? 2 : 4;
}

// Outputs that overlap the inputs or each other stay with k_direct, whose last
// kernel alone writes them and reads none: a later slab reads the inputs again and
// adds to the velocities.
static bool outputs_apart(const fss_particles *p, const fss_velocity *o)
{
    const int64_t n = p->n;
    const double *const outs[4] = {o->u, o->v, o->w, o->dvort};
    auto overlap = [n](const double *a, const double *b) {
        return std::less<const double *>()(a, b + n) && std::less<const double *>()(b, a + n);
    };
    for (int k = 0; k < 4; k++) {
        for (const double *in : {p->x, p->y, p->z, p->vort, p->area})
            if (overlap(in, outs[k])) return false;
        for (int j = 0; j < k; j++)
            if (overlap(outs[j], outs[k])) return false;
    }
    return true;
}

// The next slab from row a.r0: as many rows as leave room for their column sums
// beside the run sums of one round of resident blocks.  Its runs: one unit each
// up to two rounds; beyond that three quarters of the work in one round of long
// runs and the rest in short ones, as far as there is room for their sums.
static void sym_slab(int64_t n, int R, SymArgs &a, int64_t *blocks)
{
    const int64_t T = 256 * R, RT = 4 * R, rows = div_up(n, T), slots = R == 4 ? 768 : 1024;
    const int64_t room = SYM_BYTES / 24;
    a.K = div_up(n, 64);
    a.r1 = a.r0 + 1;
    while (a.r1 < rows && sym_col_first(a.r1 + 1, a.r0, a.K, T) + (a.r1 + 1 - a.r0 + slots) * T <= room) a.r1++;
    a.U = sym_first(a.r1, a.r0, a.K, RT);
    const int64_t cols = sym_col_first(std::min(a.r1, rows - 1), a.r0, a.K, T); // the last row has none
    const int64_t runs = (room - cols) / T - (a.r1 - a.r0);
    a.B1 = a.q1 = 0;
    if (a.U <= std::min(2 * slots, runs)) {
        a.q = 1;
    } else if (runs < 2 * slots) {
        a.q = div_up(a.U, slots);
    } else {
        a.B1 = slots;
        a.q1 = 3 * a.U / (4 * slots);
        a.q = div_up(a.U - a.B1 * a.q1, std::min<int64_t>(2 * slots, runs - slots));
    }
    *blocks = a.B1 + div_up(std::max<int64_t>(0, a.U - a.B1 * a.q1), a.q);
    a.part = a.col + 3 * cols;
}

// bytes of workspace that serve the sums of n particles and fewer (direct_bytes):
// what one slab of all rows would take, with three rounds of runs
static size_t sym_bytes(int64_t n, int R)
{
    const int64_t T = 256 * R, RT = 4 * R, rows = div_up(n, T), slots = R == 4 ? 768 : 1024, K = div_up(n, 64);
    const int64_t runs = std::min<int64_t>(sym_first(rows, 0, K, RT), 3 * slots) + rows;
    return (size_t)std::min<int64_t>(SYM_BYTES, 24 * (sym_col_first(rows - 1, 0, K, T) + runs * T));
}

template <int R>
static fss_status launch_sym(fss_ctx *ctx, const fss_particles *p, fss_velocity *out, void *buf, const RkNext &next,
                             uint64_t *ts)
{
    constexpr int64_t T = 256 * R;
    SymArgs a{};
    a.x = p->x, a.y = p->y, a.z = p->z, a.vort = p->vort, a.area = p->area;
    a.n = p->n;
    a.scale = -1.0 / (4.0 * M_PI);
    a.omega = ctx->cfg.omega;
    a.col = static_cast<double *>(buf);
    a.u = out->u, a.v = out->v, a.w = out->w, a.dvort = out->dvort;
    for (a.r0 = 0; a.r0 * T < a.n; a.r0 = a.r1) {
        int64_t blocks;
        sym_slab(a.n, R, a, &blocks);
        a.ts = a.r0 == 0 ? ts : nullptr;
        hipLaunchKernelGGL(k_direct_sym<R>, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, a);
        a.ts = ts;
        hipLaunchKernelGGL(k_sym_sum<R>, dim3((unsigned)div_up(a.n - a.r0 * T, 16)), dim3(256), 0, ctx->stream, a, next);
    }
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

// buf: at least direct_bytes() and, for the sums that sym_targets takes, sym_bytes(); ts: the call's time stamps or null
static fss_status launch_direct(fss_ctx *ctx, const fss_particles *p, const int64_t *idx, int64_t m,
                                fss_velocity *out, bool mixed, void *buf, const RkNext &next, uint64_t *ts)
{
    hipStream_t s = ctx->stream;
    const int R = sym_targets(p->n, idx, mixed);
    if (R && outputs_apart(p, out))
        return R == 2 ? launch_sym<2>(ctx, p, out, buf, next, ts) : launch_sym<4>(ctx, p, out, buf, next, ts);
    const DirectPlan P = direct_plan(p->n, m, mixed);
    DirectArgs a{p->x, p->y, p->z, p->vort, p->area, nullptr, idx, p->n, m, P.K, P.U, P.B1, P.q1, P.q, -1.0 / (4.0 * M_PI),
                 ctx->cfg.omega, static_cast<double *>(buf), out->u, out->v, out->w, out->dvort, ts};
    if (!P.split) {
        const dim3 gp((unsigned)div_up(p->n, 256));
        a.rec = buf;
        if (mixed)
            hipLaunchKernelGGL(k_pack32, gp, dim3(256), 0, s, p->x, p->y, p->z, p->vort, p->area, p->n,
                               static_cast<float4 *>(buf), ts);
        else
            hipLaunchKernelGGL(k_pack64, gp, dim3(256), 0, s, p->x, p->y, p->z, p->vort, p->area, p->n,
                               static_cast<double4 *>(buf), ts);
    }
    void (*k)(DirectArgs);
    if (mixed)
        k = !P.split ? k_direct<float, 2, 256, false> : P.R == 2 ? k_direct<float, 2, 256, true> : k_direct<float, 1, 256, true>;
    else
        k = !P.split   ? k_direct<double, 4, 64, false>
            : P.R == 4 ? k_direct<double, 4, 64, true>
            : P.R == 2 ? k_direct<double, 2, 64, true>
            : P.wt == 64 ? k_direct<double, 1, 64, true>
                         : k_direct<double, 1, 16, true>;
    hipLaunchKernelGGL(k, dim3((unsigned)P.B), dim3(256), 0, s, a);
    if (P.split)
        hipLaunchKernelGGL(k_direct_sum, dim3((unsigned)div_up(m, 16)), dim3(256), 0, s, a.part, m, 64 * P.R, P.K, P.B1, P.q1,
                           P.q, a.omega, out->u, out->v, out->w, out->dvort, next, ts);
    else if (next.mode != RkNext::NONE)
        FSS_TRY(rk4_next(ctx, next, *out)); // these kernels write every velocity where it is summed
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

fss_status velocity_direct(fss_ctx *ctx, const fss_particles *p, const int64_t *idx, int64_t m,
                           fss_velocity *out, bool force_fp64, const RkNext &next)
{
    const int64_t n = p->n;
    if (n < 1) {
        set_error("velocity_direct: n < 1");
        return FSS_ERR_INVALID;
    }
    if (!idx) m = n;
    const bool mixed = !force_fp64 && ctx->cfg.precision == FSS_MIXED;
    DevBuf &buf = ctx->direct;
    const int R = sym_targets(n, idx, mixed);
    FSS_TRY(buf.ensure(std::max(direct_bytes(n, std::max(m, n), mixed), R ? sym_bytes(n, R) : 0)));
    if (ctx->capturing) return launch_direct(ctx, p, idx, m, out, mixed, buf.p, next, nullptr);
    Timing &t = ctx->timing;
    timing_begin(t, ctx->stream);
    t.have[t.cur] = 1 << Timing::MAIN;
    FSS_TRY(launch_direct(ctx, p, idx, m, out, mixed, buf.p, next, t.slot()));
    t.valid = true;
    return FSS_OK;
}

// ------------------------------------------------------------------
// allocation-free variant: the partial sums or packed source records live in
// a file-scope device array instead of the context's workspace
// ------------------------------------------------------------------
// One copy per GPU, held until the process ends.  Every call on a GPU writes
// that GPU's copy, so calls that overlap on one GPU (two streams, two threads)
// race; calls in one stream order are safe.  Nothing in it needs clearing: a
// call reads only what it wrote.
static __device__ __align__(256) unsigned char scratch[DIRECT_SCRATCH];

constexpr int SCRATCH_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch[SCRATCH_MAX_DEVICES] = {};

fss_status direct_scratch_setup(int device)
{
    if (device < 0 || device >= SCRATCH_MAX_DEVICES) {
        set_error("direct scratch: device index beyond " + std::to_string(SCRATCH_MAX_DEVICES));
        return FSS_ERR_INVALID;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device]) return FSS_OK;
    int cur = -1;
    FSS_HIP(hipGetDevice(&cur));
    if (cur != device) {
        set_error("direct scratch: set-up needs its device current");
        return FSS_ERR_STATE;
    }
    void *ptr = nullptr;
    FSS_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) {
        set_error("direct scratch: no device address");
        return FSS_ERR_HIP;
    }
    g_scratch[device] = ptr;
    return FSS_OK;
}

fss_status velocity_direct_noalloc(fss_ctx *ctx, const fss_particles *p, fss_velocity *out)
{
    const int64_t n = p->n;
    const bool mixed = ctx->cfg.precision == FSS_MIXED;
    const size_t rec = mixed ? sizeof(float4) : sizeof(double4);
    if (n < 1 || (size_t)n > FSS_DIRECT_SCRATCH_BYTES / rec) {
        set_error("velocity_direct_noalloc: n must be in [1, " +
                  std::to_string(FSS_DIRECT_SCRATCH_BYTES / rec) + "] in " + (mixed ? "mixed" : "FP64") +
                  " precision (" + std::to_string(FSS_DIRECT_SCRATCH_BYTES >> 20) + " MiB of records), got " +
                  std::to_string(n));
        return FSS_ERR_INVALID;
    }
    const int dev = ctx->cfg.device;
    void *buf = (dev >= 0 && dev < SCRATCH_MAX_DEVICES) ? g_scratch[dev] : nullptr;
    if (!buf) {
        set_error("velocity_direct_noalloc: scratch of device " + std::to_string(dev) + " not set up");
        return FSS_ERR_STATE;
    }
    return launch_direct(ctx, p, nullptr, n, out, mixed, buf, RkNext{}, nullptr);
}

} // namespace fss
