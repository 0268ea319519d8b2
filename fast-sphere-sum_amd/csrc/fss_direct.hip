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
// Bound by FP64 issue (17 four-cycle slots a pair at four targets a lane: 822 us
// at N = 40,009, 1.95e12 pairs/s at about 2 GHz).  One target a lane, one block
// per 256 targets and a reciprocal with two Newton steps per pair took 2,036
// us there, 525 us at N = 10,242 (41 blocks on 256 CUs; now 79) and 42.6 ms for
// 10,000 targets of N = 655,362 (now 3.4).
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
#include <mutex>

#include "fss_internal.h"

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

__device__ inline void direct_source(const DirectArgs &a, int64_t j, double4 &s)
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
                                                    double *dvort, uint64_t *ts)
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
        u[r] = red[0][0][tl];
        v[r] = red[1][0][tl];
        w[r] = red[2][0][tl];
        dvort[r] = -2 * omega * red[2][0][tl];
    }
    stamp_end(ts);
}

struct DirectPlan {
    int R, wt; // targets per lane, sources per wave tile
    bool split;
    int64_t K, G, U, B1, q1, q, B;
    size_t bytes; // partials or packed records
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

static DirectPlan direct_plan(int64_t n, int64_t m, bool mixed)
{
    DirectPlan p{};
    const DirectLayout *lay = mixed ? kDirect32 : kDirect64;
    const int nl = mixed ? 2 : 4;
    p.split = div_up(m, 256) < DIRECT_SPLIT_GROUPS;
    int pick = nl - 1;
    double best = INFINITY;
    for (int k = 0; k < nl && p.split; k++) {
        const double t = lay[k].lone + (double)(div_up(m, 64 * lay[k].R) * 64 * lay[k].R) * (double)n / lay[k].rate;
        if (t < best) {
            best = t;
            pick = k;
        }
    }
    p.R = lay[pick].R;
    p.wt = lay[pick].wt;
    p.K = div_up(n, p.wt);
    p.G = div_up(m, 64 * p.R);
    p.U = p.G * p.K;
    if (!p.split) {
        p.q = p.K;
        p.B = p.G;
        p.bytes = (mixed ? sizeof(float4) : sizeof(double4)) * (size_t)n;
        return p;
    }
    // Runs, in quads of units (one per wave): up to about two rounds of the
    // 1,024 resident blocks one quad each; above, three quarters of the work in
    // one round of long runs and the rest in short ones, so that the blocks that
    // end last are short (equal runs in two rounds: 872 us at N = 40,009, in
    // four 841).  The partials of all of them stay within 30 MiB.
    const int64_t V = div_up(p.U, 4), slots = 1024;
    const int64_t most = ((int64_t)30 << 20) / (1536 * p.R) - p.G;
    if (V <= std::min<int64_t>(2 * slots, most)) {
        p.q = 4;
    } else {
        p.B1 = slots;
        p.q1 = 4 * (3 * V / (4 * slots));
        const int64_t rest = V - p.B1 * (p.q1 / 4);
        p.q = 4 * div_up(rest, std::min<int64_t>(3 * slots, most - slots));
    }
    p.B = p.B1 + div_up(std::max<int64_t>(0, p.U - p.B1 * p.q1), p.q);
    p.bytes = sizeof(double) * 3 * 64 * p.R * (size_t)(p.B + p.G);
    return p;
}

// buf: at least direct_plan().bytes; ts: the call's time stamps or null
static fss_status launch_direct(fss_ctx *ctx, const fss_particles *p, const int64_t *idx, int64_t m,
                                fss_velocity *out, bool mixed, void *buf, uint64_t *ts)
{
    hipStream_t s = ctx->stream;
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
                           P.q, a.omega, out->u, out->v, out->w, out->dvort, ts);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

fss_status velocity_direct(fss_ctx *ctx, const fss_particles *p, const int64_t *idx, int64_t m,
                           fss_velocity *out, bool force_fp64)
{
    const int64_t n = p->n;
    if (n < 1) {
        set_error("velocity_direct: n < 1");
        return FSS_ERR_INVALID;
    }
    if (!idx) m = n;
    const bool mixed = !force_fp64 && ctx->cfg.precision == FSS_MIXED;
    DevBuf &buf = ctx->direct;
    FSS_TRY(buf.ensure(direct_plan(n, m, mixed).bytes));
    if (ctx->capturing) return launch_direct(ctx, p, idx, m, out, mixed, buf.p, nullptr);
    Timing &t = ctx->timing;
    timing_begin(t, ctx->stream);
    t.have[t.cur] = 1 << Timing::MAIN;
    FSS_TRY(launch_direct(ctx, p, idx, m, out, mixed, buf.p, t.slot()));
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
static __device__ __align__(256) unsigned char scratch[FSS_DIRECT_SCRATCH_BYTES];

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
                  " precision (" + std::to_string(FSS_DIRECT_SCRATCH_BYTES >> 20) + " MiB of scratch), got " +
                  std::to_string(n));
        return FSS_ERR_INVALID;
    }
    const int dev = ctx->cfg.device;
    void *buf = (dev >= 0 && dev < SCRATCH_MAX_DEVICES) ? g_scratch[dev] : nullptr;
    if (!buf) {
        set_error("velocity_direct_noalloc: scratch of device " + std::to_string(dev) + " not set up");
        return FSS_ERR_STATE;
    }
    return launch_direct(ctx, p, nullptr, n, out, mixed, buf, nullptr);
}

} // namespace fss
