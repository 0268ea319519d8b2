// fss_sal_tree.hip -- SAL convolution by the barycentric-Lagrange treecode.
//
// eta_SAL(x_i) = sum_j G(s_ij) eta_j A_j, j = i included (salpotential,
// SAL/GFnewtest.ipynb:9934-9949), s = |x_i - x_j| / 2, on the same tree,
// interaction list and evaluation plan as the velocity (BLTC mode): near
// items evaluate G directly, proxy items evaluate G between the target
// node's proxies and its class-B sources (particles, or source proxies that
// carry the modified charges of the upward pass), the interpolant of every
// target node is solved and evaluated at its particles.  Scalar kernel, FP64
// records; G is one of
//   KIND 0  the tabulated series (cubic interpolation, the fast fallback),
//   KIND 1  the learned kernel (analytic singular part + network),
//   KIND 2  the series itself by Clenshaw summation (the accuracy reference).
#include <hip/hip_runtime.h>

#include "fss_geom.h"
#include "fss_sal_dev.h"

namespace fss {

namespace {

// sources staged at a time: 4.6 KiB a one-wave block for the table, eight waves per
// SIMD in place of four
constexpr int sal_chunk_size(int kind) { return kind == 2 ? 256 : 128; }

template <int D> constexpr int npts_s() { return (D + 1) * (D + 2) / 2; }

struct KernelArgs {
    SalTab tab;
    const float *P;
    const MlpOp *mlp;   // the network's parameters in the form of the matrix-core evaluation
    double A, mu, sigma, g0;
    float log_smin, inv_span;
    const double *c;
    int N;
    uint64_t *ts_near, *ts_proxy, *ts; // time stamps, or null
};

__device__ inline double dist2(const double4 &a, const double4 &b)
{
    double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    return dx * dx + dy * dy + dz * dz;
}

__device__ inline double half_dist(const double4 &a, const double4 &b) { return 0.5 * sqrt(dist2(a, b)); }

// the series kernels (KIND 0: table, 2: Clenshaw); the learned kernel has
// its own matrix-core kernels below
template <int KIND> __device__ inline double gfun(const KernelArgs &k, const double4 &a, const double4 &b)
{
    static_assert(KIND == 0 || KIND == 2, "series kernels only");
    const double q = dist2(a, b);
    if (KIND == 0) return table_eval_dist2(k.tab, q);
    const double s = 0.5 * sqrt(q);
    return legendre_sum(k.c, k.N, 1.0 - 2.0 * s * s);
}

// the staged sources ph, ph + P, ... below m against the R targets of a lane
template <int KIND, int R>
__device__ inline void sal_chunk(const KernelArgs &ka, const double4 *xt, const double4 *lds, int ph, int P, int m,
                                 double *acc)
{
    for (int k = ph; k < m; k += P) {
        const double4 s = lds[k];
#pragma unroll
        for (int q = 0; q < R; q++) acc[q] = fma(gfun<KIND>(ka, xt[q], s), s.w, acc[q]);
    }
}

// Targets (proxies) per lane.  The table lookups bound these kernels: every lane
// reads its own two lines from L1, one lookup a cycle and CU (level-8 grid, degree
// 3: 2.26 lookups a near pair, 1.02 a cycle), so several targets a lane help by
// what they put in flight and by the lanes that one target a lane leaves idle (33 to
// 64 targets: the lanes beyond them; level-8 grid, near field with 1 / 2 / 3 / 4 / 5 /
// 6 targets a lane: call of 4.35 / 3.88 / 4.35 / 3.63 / 3.95 / 4.84 ms).  Proxies: all of a
// node's up to degree 3, a third beyond (call at degree 3 with 1 / 2 / 5 / 10: 3.63 / 3.51 /
// 3.38 / 3.27 ms; degree 4 with 1 / 3 / 5 / 8: 5.96 / 6.33 / 5.73 / 5.82; degree 5 with 1 / 3 / 6 /
// 7: 9.97 / 10.63 / 12.61 / 9.63).  Contiguous runs of items per XCD are slower (6.1
// against 4.3 ms), and so are two lanes sharing each window of the table (half the
// loads' lines, but the exchange costs more: 4.0 ms).
// The Clenshaw series is arithmetic alone, and the targets that fill up a lane's
// count cost as much as others: one a lane (200,003 particles, 6 levels, 65 terms,
// degree 1 / 3 / 5: 8.9 / 21.4 / 59.0 ms; with the table's counts and chunks 10.6 / 23.7 /
// 69.4).
constexpr int sal_near_r(int kind) { return kind == 2 ? 1 : 4; }
constexpr int sal_proxy_r(int kind, int pp) { return kind == 2 ? 1 : pp <= 10 ? pp : pp / 3; }

// near field: one wave per near item, R targets per lane and phase; the
// item's source list (the self ranges too: j = i is part of the sum) staged in
// LDS chunks, every chunk's loads independent
template <int KIND, int R>
__global__ void __launch_bounds__(64) k_sal_near(const NearItem *__restrict__ items,
                                                 const int32_t *__restrict__ near_src,
                                                 const double4 *__restrict__ src, KernelArgs ka, double *out)
{
    stamp_start(ka.ts_near, Timing::MAIN);
    constexpr int NCH_S = sal_chunk_size(KIND);
    __shared__ double4 lds[NCH_S];
    __shared__ double red[64 * R];
    const NearItem it = items[blockIdx.x];
    const int lane = threadIdx.x;
    const int cnt = it.tgt_cnt;
    const int T = (cnt + R - 1) / R, P = 64 / T;
    const int ph = lane / T, tl = lane - ph * T;
    const bool act = ph < P;
    double4 xt[R];
    double acc[R] = {};
#pragma unroll
    for (int q = 0; q < R; q++) {
        // a missing target repeats the lane's first: the same table cells
        xt[q] = src[it.tgt_start + (act ? (tl + q * T < cnt ? tl + q * T : tl) : 0)];
    }
    const int32_t *list = near_src + it.src_off;
    const int total = it.n_other + it.n_self;
    for (int base = 0; base < total; base += NCH_S) {
        const int m = min(NCH_S, total - base);
#pragma unroll
        for (int s = 0; s < NCH_S / 64; s++)
            if (lane + 64 * s < m) lds[lane + 64 * s] = src[list[base + lane + 64 * s]];
        __syncthreads();
        if (act) sal_chunk<KIND, R>(ka, xt, lds, ph, P, m, acc);
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < R; q++) red[64 * q + lane] = acc[q];
    __syncthreads();
    if (lane < cnt) {
        const int q = lane / T, g = lane - q * T;
        double a = 0.0;
        for (int h = 0; h < P; h++) a += red[64 * q + h * T + g];
        out[it.out_base + lane] = a;
    }
}

// proxy values: one wave per proxy item, R proxies per lane, phases as in
// k_sal_near; the item's source list staged in LDS chunks
template <int KIND, int D, int R>
__global__ void __launch_bounds__(64) k_sal_proxy(const ProxyItem *__restrict__ items,
                                                  const int64_t *__restrict__ far_off,
                                                  const int32_t *__restrict__ far_src,
                                                  const double4 *__restrict__ src, int64_t p0, KernelArgs ka,
                                                  double *phi)
{
    stamp_start(ka.ts_proxy, Timing::MAIN);
    constexpr int PP = npts_s<D>();
    constexpr int T = (PP + R - 1) / R, P = 64 / T;
    constexpr int NCH_S = sal_chunk_size(KIND);
    __shared__ double4 lds[NCH_S];
    __shared__ double red[64 * R];
    const int64_t item = blockIdx.x;
    const ProxyItem it = items[item];
    const int lane = threadIdx.x;
    const int ph = lane / T, tl = lane - ph * T;
    const bool act = ph < P;
    double4 yk[R];
    double acc[R] = {};
#pragma unroll
    for (int q = 0; q < R; q++) {
        yk[q] = src[p0 + (int64_t)it.node * PP + (act ? (tl + q * T < PP ? tl + q * T : tl) : 0)];
    }
    const int64_t o0 = far_off[item];
    const int total = (int)(far_off[item + 1] - o0);
    const int32_t *list = far_src + o0;
    for (int base = 0; base < total; base += NCH_S) {
        const int m = min(NCH_S, total - base);
#pragma unroll
        for (int s = 0; s < NCH_S / 64; s++)
            if (lane + 64 * s < m) lds[lane + 64 * s] = src[list[base + lane + 64 * s]];
        __syncthreads();
        if (act) sal_chunk<KIND, R>(ka, yk, lds, ph, P, m, acc);
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < R; q++) red[64 * q + lane] = acc[q];
    __syncthreads();
    if (lane < PP) {
        const int q = lane / T, g = lane - q * T;
        double a = 0.0;
        for (int h = 0; h < P; h++) a += red[64 * q + h * T + g];
        phi[item * PP + lane] = a;
    }
}

// ------------------------------------------------------------------
// learned kernel on the matrix cores
// ------------------------------------------------------------------
// Four items per block (one per wave) share the network parameters staged in
// LDS; every wave stages its own source chunks.  The lanes keep the (target
// or proxy, phase) layout of the kernels above, but the source loop runs a
// wave-uniform number of trips so that every network evaluation (64 pairs at
// once) sees the whole wave; lanes without a pair in a trip evaluate a dummy
// input and add nothing.
constexpr int NCH_M = 128;

__device__ inline void sal_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// G(s) of the learned kernel from the network output y (s = 0: self term)
__device__ inline double learned_g(const KernelArgs &k, double s, float y)
{
    return s > 0.0 ? k.A * (0.5 / s - 1.0) + k.mu + k.sigma * (double)y : k.g0;
}

__global__ void __launch_bounds__(256) k_sal_near_mlp(const NearItem *__restrict__ items, int64_t nitems,
                                                      const int32_t *__restrict__ near_src,
                                                      const double4 *__restrict__ src, KernelArgs ka, double *out)
{
    stamp_start(ka.ts_near, Timing::MAIN);
    __shared__ MlpOp Ml;
    __shared__ double4 stage[4][NCH_M];
    __shared__ double red[4][64];
    mlp_stage(Ml, ka.mlp);
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t item = (int64_t)blockIdx.x * 4 + wave;
    if (item >= nitems) return; // the whole wave; no block barrier follows
    double4 *lds = stage[wave];
    const NearItem it = items[item];
    const int lane = threadIdx.x & 63;
    const int cnt = it.tgt_cnt;
    const int P = 64 / cnt;
    const int ph = lane / cnt, tl = lane - ph * cnt;
    const bool act = ph < P;
    const double4 xt = src[it.tgt_start + (act ? tl : 0)];
    double acc = 0.0;
    const int32_t *list = near_src + it.src_off;
    const int total = it.n_other + it.n_self;
    for (int base = 0; base < total; base += NCH_M) {
        const int m = min(NCH_M, total - base);
#pragma unroll
        for (int s = 0; s < NCH_M / 64; s++)
            if (lane + 64 * s < m) lds[lane + 64 * s] = src[list[base + lane + 64 * s]];
        sal_wave_sync();
        const int trips = (m + P - 1) / P;
        for (int t = 0; t < trips; t++) {
            const int k = ph + t * P;
            const bool ok = act && k < m;
            const double4 sv = lds[ok ? k : 0];
            const double s = half_dist(xt, sv);
            const float y = mlp_wave64(Ml, mlp_input(s > 0.0 ? s : 1.0, ka.log_smin, ka.inv_span));
            if (ok) acc = fma(learned_g(ka, s, y), sv.w, acc);
        }
        sal_wave_sync();
    }
    red[wave][lane] = acc;
    sal_wave_sync();
    if (ph == 0 && act) {
        double a = 0.0;
        for (int h = 0; h < P; h++) a += red[wave][h * cnt + tl];
        out[it.out_base + tl] = a;
    }
}

template <int D>
__global__ void __launch_bounds__(256) k_sal_proxy_mlp(const ProxyItem *__restrict__ items, int64_t nitems,
                                                       const int64_t *__restrict__ far_off,
                                                       const int32_t *__restrict__ far_src,
                                                       const double4 *__restrict__ src, int64_t p0, KernelArgs ka,
                                                       double *phi)
{
    stamp_start(ka.ts_proxy, Timing::MAIN);
    constexpr int PP = npts_s<D>();
    constexpr int P = 64 / PP;
    __shared__ MlpOp Ml;
    __shared__ double4 stage[4][NCH_M];
    __shared__ double red[4][64];
    mlp_stage(Ml, ka.mlp);
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t item = (int64_t)blockIdx.x * 4 + wave;
    if (item >= nitems) return;
    double4 *lds = stage[wave];
    const ProxyItem it = items[item];
    const int lane = threadIdx.x & 63;
    const int ph = lane / PP, k = lane - ph * PP;
    const bool act = ph < P;
    const double4 yk = src[p0 + (int64_t)it.node * PP + (act ? k : 0)];
    double acc = 0.0;
    const int64_t o0 = far_off[item];
    const int total = (int)(far_off[item + 1] - o0);
    const int32_t *list = far_src + o0;
    for (int base = 0; base < total; base += NCH_M) {
        const int m = min(NCH_M, total - base);
#pragma unroll
        for (int s = 0; s < NCH_M / 64; s++)
            if (lane + 64 * s < m) lds[lane + 64 * s] = src[list[base + lane + 64 * s]];
        sal_wave_sync();
        const int trips = (m + P - 1) / P;
        for (int t = 0; t < trips; t++) {
            const int kk = ph + t * P;
            const bool ok = act && kk < m;
            const double4 sv = lds[ok ? kk : 0];
            const double s = half_dist(yk, sv);
            const float y = mlp_wave64(Ml, mlp_input(s > 0.0 ? s : 1.0, ka.log_smin, ka.inv_span));
            if (ok) acc = fma(learned_g(ka, s, y), sv.w, acc);
        }
        sal_wave_sync();
    }
    red[wave][lane] = acc;
    sal_wave_sync();
    if (ph == 0 && act) {
        double a = 0.0;
        for (int h = 0; h < P; h++) a += red[wave][h * PP + k];
        phi[item * PP + k] = a;
    }
}

// sum the chunks of every interpolant slot in order and solve V alpha = phi
// (one right-hand side; the row interchanges applied while summing)
template <int D>
__global__ void __launch_bounds__(128) k_sal_solve(const ProxySlot *__restrict__ slots, int64_t nslot, const double *__restrict__ phi,
                            const double *__restrict__ lu, const int32_t *__restrict__ perm, double *alpha)
{
    constexpr int P = npts_s<D>();
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nslot) return;
    const ProxySlot sl = slots[q];
    double b[P];
#pragma unroll
    for (int k = 0; k < P; k++) b[k] = 0.0;
    for (int part = sl.part_beg; part < sl.part_end; part++)
#pragma unroll
        for (int k = 0; k < P; k++) b[k] += phi[(int64_t)part * P + perm[k]];
#pragma unroll
    for (int k = 0; k < P; k++)
#pragma unroll
        for (int r = k + 1; r < P; r++) b[r] = b[r] - b[k] * lu[r + k * P];
#pragma unroll
    for (int k = P - 1; k >= 0; k--) {
        b[k] = b[k] / lu[k + k * P];
#pragma unroll
        for (int r = 0; r < k; r++) b[r] = b[r] - b[k] * lu[r + k * P];
    }
    for (int k = 0; k < P; k++) alpha[q * P + k] = b[k];
}

template <int D>
__device__ inline double sal_interp(const double *__restrict__ tinv, const double *__restrict__ alpha, int32_t g,
                                    int32_t sl, const double *pt)
{
    constexpr int P = npts_s<D>();
    const double *R = tinv + 9 * (int64_t)g;
    double c[3];
    for (int m = 0; m < 3; m++) c[m] = fma(R[3 * m], pt[0], fma(R[3 * m + 1], pt[1], R[3 * m + 2] * pt[2]));
    const double is = 1.0 / (c[0] + c[1] + c[2]);
    const double s = c[0] * is, t = c[1] * is;
    double sp[D + 1], tp[D + 1];
    sp[0] = tp[0] = 1.0;
    for (int k = 1; k <= D; k++) {
        sp[k] = sp[k - 1] * s;
        tp[k] = tp[k - 1] * t;
    }
    const double *al = alpha + (int64_t)sl * P;
    double v = 0.0;
    for (int i = 0; i <= D; i++)
        for (int j = 0; j <= i; j++) v = fma(sp[i - j] * tp[j], al[i * (i + 1) / 2 + j], v);
    return v;
}

// per main record (tree order): near slots of its main path + interpolants of
// the nodes on it; memberships outside the main path from the per-level maps
template <int D>
__global__ void k_sal_combine(const int32_t *__restrict__ recid, const int32_t *__restrict__ recnode,
                              const uint8_t *__restrict__ rinfo, const int4 *__restrict__ nrange,
                              const int32_t *__restrict__ oslot, const int32_t *__restrict__ node_slot,
                              const int32_t *__restrict__ nodeof, const int32_t *__restrict__ inv_active,
                              const double *__restrict__ alpha, const double *__restrict__ tinv,
                              const double4 *__restrict__ src, const Instance *__restrict__ inst, int ninst,
                              int64_t nrec, const double *__restrict__ out, double *acc)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrec) return;
    int lo = 0, hi = ninst - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) / 2;
        if (inst[mid].rbase <= i) lo = mid;
        else hi = mid - 1;
    }
    const Instance I = inst[lo];
    if (i - I.rbase >= I.n) return;
    const double4 r = src[i];
    const double pt[3] = {r.x, r.y, r.z};
    const int info = rinfo[i];
    const int e = info & 0x7f;
    double a = 0.0;
    if (e > 0) {
        const int ld = e - 1;
        const int64_t locd = recnode[i] - I.nbase - fssg::level_offset(ld);
        for (int l = 0; l < e; l++) {
            const int32_t g = (int32_t)(I.nbase + fssg::level_offset(l) + (locd >> (2 * (ld - l))));
            const int32_t gu = __builtin_amdgcn_readfirstlane(g);
            if (__all(g == gu)) { // node shared by the wave: scalar loads
                const int32_t os = oslot[gu];
                if (os >= 0) a += out[os + (i - nrange[gu].x)];
                const int32_t sl = node_slot[gu];
                if (sl >= 0) a += sal_interp<D>(tinv, alpha, gu, sl, pt);
            } else {
                const int32_t os = oslot[g];
                if (os >= 0) a += out[os + (i - nrange[g].x)];
                // a few nodes per wave: one pass per distinct node through
                // scalar loads of its interpolant
                const int32_t sl = node_slot[g];
                bool todo = sl >= 0;
                uint64_t msk;
                while ((msk = __ballot(todo)) != 0) {
                    const int fl = __builtin_ctzll(msk);
                    const int32_t gs = __builtin_amdgcn_readlane(g, fl), ss = __builtin_amdgcn_readlane(sl, fl);
                    if (todo && g == gs) {
                        a += sal_interp<D>(tinv, alpha, gs, ss, pt);
                        todo = false;
                    }
                }
            }
        }
    }
    if (info & 0x80) {
        const int64_t li = recid[i] - I.pbase;
        for (int l = e; l < I.L; l++) {
            const int64_t at = I.loff + (int64_t)l * I.n + li;
            const int32_t g = nodeof[at];
            if (g < 0) continue;
            const int32_t pos = inv_active[at];
            if (pos >= 0) a += out[pos];
            const int32_t sl = node_slot[g];
            if (sl >= 0) a += sal_interp<D>(tinv, alpha, g, sl, pt);
        }
    }
    acc[i] = a;
}

__global__ void k_sal_scatter(const int32_t *__restrict__ ipos, int64_t n, const double *__restrict__ acc,
                              double *out, uint64_t *ts)
{
    int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id < n) out[id] = acc[ipos[id]];
    stamp_end(ts);
}

template <int KIND, int D> fss_status run(fss_ctx *ctx, const KernelArgs &ka, double *result)
{
    Tree &T = ctx->tree;
    hipStream_t s = ctx->stream;
    constexpr int p = npts_s<D>();
    const int64_t p0 = T.p0;
    const double4 *src = T.src64.as<double4>();
    FSS_TRY(ctx->out3.ensure(sizeof(double) * std::max<int64_t>(1, T.nslot_out)));
    FSS_TRY(ctx->phi.ensure(sizeof(double) * p * std::max<int64_t>(1, T.n_proxy)));
    FSS_TRY(ctx->alpha.ensure(sizeof(double) * p * std::max<int64_t>(1, T.n_slot)));
    FSS_TRY(ctx->acc3.ensure(sizeof(double) * std::max<int64_t>(1, p0)));
    if constexpr (KIND == 1) {
        // the learned kernel: network evaluations on the matrix cores, four
        // items per block
        if (T.n_near > 0)
            hipLaunchKernelGGL(k_sal_near_mlp, dim3((unsigned)div_up(T.n_near, 4)), dim3(256), 0, s,
                               T.near_items.as<NearItem>(), T.n_near, T.near_src.as<int32_t>(), src, ka,
                               ctx->out3.as<double>());
        if (T.n_proxy > 0)
            hipLaunchKernelGGL((k_sal_proxy_mlp<D>), dim3((unsigned)div_up(T.n_proxy, 4)), dim3(256), 0, s,
                               T.proxy_items.as<ProxyItem>(), T.n_proxy, T.far_off.as<int64_t>(),
                               T.far_src.as<int32_t>(), src, p0, ka, ctx->phi.as<double>());
    } else {
        constexpr int RN = sal_near_r(KIND), RF = sal_proxy_r(KIND, npts_s<D>());
        if (T.n_near > 0)
            hipLaunchKernelGGL((k_sal_near<KIND, RN>), dim3((unsigned)T.n_near), dim3(64), 0, s,
                               T.near_items.as<NearItem>(), T.near_src.as<int32_t>(), src, ka, ctx->out3.as<double>());
        if (T.n_proxy > 0)
            hipLaunchKernelGGL((k_sal_proxy<KIND, D, RF>), dim3((unsigned)T.n_proxy), dim3(64), 0, s,
                               T.proxy_items.as<ProxyItem>(), T.far_off.as<int64_t>(), T.far_src.as<int32_t>(), src,
                               p0, ka, ctx->phi.as<double>());
    }
    if (T.n_slot > 0)
        hipLaunchKernelGGL((k_sal_solve<D>), dim3((unsigned)div_up(T.n_slot, 128)), dim3(128), 0, s,
                           T.proxy_slots.as<ProxySlot>(), T.n_slot, ctx->phi.as<double>(), ctx->d_lu.as<double>(),
                           ctx->d_perm.as<int32_t>(), ctx->alpha.as<double>());
    hipLaunchKernelGGL((k_sal_combine<D>), dim3((unsigned)div_up(p0, 256)), dim3(256), 0, s, T.recid.as<int32_t>(),
                       T.recnode.as<int32_t>(), T.rinfo.as<uint8_t>(), T.nrange.as<int4>(), T.oslot.as<int32_t>(),
                       T.node_slot.as<int32_t>(), T.nodeof.as<int32_t>(), T.inv_active.as<int32_t>(),
                       ctx->alpha.as<double>(), T.d_tinv, src, T.inst.as<Instance>(), T.ninst, p0,
                       ctx->out3.as<double>(), ctx->acc3.as<double>());
    hipLaunchKernelGGL(k_sal_scatter, dim3((unsigned)div_up(T.n, 256)), dim3(256), 0, s, T.ipos.as<int32_t>(), T.n,
                       ctx->acc3.as<double>(), result, ka.ts);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

template <int KIND> fss_status run_kind(fss_ctx *ctx, const KernelArgs &ka, double *result)
{
    switch (ctx->interp.degree) {
    case 1: return run<KIND, 1>(ctx, ka, result);
    case 2: return run<KIND, 2>(ctx, ka, result);
    case 3: return run<KIND, 3>(ctx, ka, result);
    case 4: return run<KIND, 4>(ctx, ka, result);
    case 5: return run<KIND, 5>(ctx, ka, result);
    default: set_error("sal treecode: degree 1..5"); return FSS_ERR_INVALID;
    }
}

} // namespace

fss_status sal_tree(fss_ctx *ctx, const fss_particles *pp, int kind, double *out)
{
    Tree &T = ctx->tree;
    Sal &S = ctx->sal;
    if (!T.built) return set_error("sal treecode: build the tree first"), FSS_ERR_STATE;
    if (ctx->cfg.eval_mode != FSS_EVAL_BLTC) return set_error("sal treecode: needs eval_mode BLTC"), FSS_ERR_STATE;
    if (pp->n != T.n) return set_error("particle count differs from the tree's"), FSS_ERR_INVALID;
    if (!S.c.p) return set_error("sal: series not set"), FSS_ERR_STATE;
    if (kind == 1 && !S.has_mlp) return set_error("sal: no network"), FSS_ERR_STATE;
    if (kind < 0 || kind > 2) return set_error("sal: kind 0 (table), 1 (learned) or 2 (series)"), FSS_ERR_INVALID;
    if (kind == 1) FSS_TRY(sal_mlp_prepare(ctx));
    KernelArgs ka;
    ka.tab = sal_tab(S.tab.as<double>(), S.M);
    ka.P = S.P.as<float>();
    ka.mlp = S.mlpop.as<MlpOp>();
    ka.A = S.A;
    ka.mu = S.mu;
    ka.sigma = S.sigma;
    ka.g0 = S.g0;
    ka.log_smin = (float)std::log(S.s_min);
    ka.inv_span = (float)(1.0 / -std::log(S.s_min));
    ka.c = S.c.as<double>();
    ka.N = S.nmax;
    ka.ts = ka.ts_near = ka.ts_proxy = nullptr;
    if (!ctx->capturing) {
        Timing &t = ctx->timing;
        timing_begin(t, ctx->stream);
        t.have[t.cur] = T.n_near > 0 || T.n_proxy > 0 ? 1 << Timing::MAIN : 0;
        ka.ts = t.slot();
        (T.n_near > 0 ? ka.ts_near : ka.ts_proxy) = ka.ts;
    }
    FSS_TRY(tree_sources64(ctx, pp, ka.ts)); // records w = eta A and the modified charges
    fss_status st = kind == 0 ? run_kind<0>(ctx, ka, out) : kind == 1 ? run_kind<1>(ctx, ka, out)
                                                                    : run_kind<2>(ctx, ka, out);
    if (ka.ts) ctx->timing.valid = true;
    return st;
}

} // namespace fss
