// fss_rk4.hip -- RK4 time step with projection onto the sphere, FP64 on the
// device, and its hipGraph.
//
// Intended semantics of the reference driver (Old-BVE-code/new_dynamics.cpp:142-238;
// its shipped text uses undeclared stage buffers):
//   k1 = f(y); y1 = proj(y + dt/2 k1); k2 = f(y1); y2 = proj(y + dt/2 k2);
//   k3 = f(y2); y3 = proj(y + dt k3); k4 = f(y3);
//   y += dt/6 (k1 + 2 k2 + 2 k3 + k4); proj(y)
// The updates are taken by the last kernel of each evaluation (fss_rk4_dev.h).
// The tree is the t = 0 tree (new_dynamics.cpp:84-88 builds it once).
#include <cmath>

#include "fss_internal.h"
#include "fss_rk4_dev.h"

namespace fss {

__global__ void k_rk4_next(RkNext r, fss_velocity k)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < r.n) rk_next(r, i, k.u[i], k.v[i], k.w[i], k.dvort[i]);
}

fss_status rk4_next(fss_ctx *ctx, const RkNext &r, const fss_velocity &k)
{
    hipLaunchKernelGGL(k_rk4_next, dim3((unsigned)div_up(r.n, 256)), dim3(256), 0, ctx->stream, r, k);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

// Tree order: with a tree the step runs on copies in the order of the source
// records, so that every stage gathers its records and writes its velocities
// and states in order.  Random particle orders paid for it in each of the four
// stages (3.05 M particles, 24 instances: gather 183 and combine 285 us a stage in
// the caller's order, 31 and 154 in tree order).
__global__ void k_rk4_load(const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
                           const double *__restrict__ vo, const double *__restrict__ area,
                           const int32_t *__restrict__ recid, int64_t n, double *t)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t id = recid[i];
    t[i] = x[id];
    t[n + i] = y[id];
    t[2 * n + i] = z[id];
    t[3 * n + i] = vo[id];
    t[4 * n + i] = area[id];
}

__global__ void k_rk4_store(const double *__restrict__ t, const int32_t *__restrict__ recid, int64_t n, double *x,
                            double *y, double *z, double *vo)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t id = recid[i];
    x[id] = t[i];
    y[id] = t[n + i];
    z[id] = t[2 * n + i];
    vo[id] = t[3 * n + i];
}

__global__ void k_project(double *x, double *y, double *z, double *vo, int64_t n, double omega)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double a = x[i], b = y[i], c = z[i], d = vo[i];
    project_one(a, b, c, d, omega);
    x[i] = a;
    y[i] = b;
    z[i] = c;
    vo[i] = d;
}

fss_status project_points(fss_ctx *ctx, double *x, double *y, double *z, double *vort, int64_t n)
{
    hipLaunchKernelGGL(k_project, dim3((unsigned)div_up(n, 256)), dim3(256), 0, ctx->stream, x, y, z,
                       vort, n, ctx->cfg.omega);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

// the state a step works on: the caller's arrays, or their copies in tree order
struct State {
    double *x, *y, *z, *vort;
    const double *area;
    bool tree_order;
};

static fss_status eval(fss_ctx *ctx, const double *x, const double *y, const double *z,
                       const double *vo, const State &S, int64_t n, double *k, int use_tree, const RkNext &next)
{
    fss_particles p{x, y, z, vo, S.area, n};
    fss_velocity o{k, k + n, k + 2 * n, k + 3 * n};
    if (use_tree) return velocity_tree(ctx, &p, &o, S.tree_order, next);
    return velocity_direct(ctx, &p, nullptr, n, &o, false, next);
}

static fss_status step(fss_ctx *ctx, const State &S, int64_t n, double dt, int use_tree)
{
    double *K = ctx->rk_k.as<double>(), *Y = ctx->rk_y.as<double>();
    const double fac[4] = {dt / 2, dt / 2, dt, dt / 6};
    for (int st = 0; st < 4; st++) {
        const RkNext next{st < 3 ? RkNext::STAGE : RkNext::STEP, S.x, S.y, S.z, S.vort, K, Y, n, fac[st], ctx->cfg.omega};
        if (st == 0) FSS_TRY(eval(ctx, S.x, S.y, S.z, S.vort, S, n, K, use_tree, next));
        else FSS_TRY(eval(ctx, Y, Y + n, Y + 2 * n, Y + 3 * n, S, n, K + 4 * n * st, use_tree, next));
    }
    return FSS_OK;
}

// workspace of a run on the caller's arrays, and its state (loaded)
static fss_status begin(fss_ctx *ctx, double *x, double *y, double *z, double *vort, const double *area, int64_t n,
                        int use_tree, State &S)
{
    const Tree &T = ctx->tree;
    if (use_tree && (!T.built || T.n != n)) {
        set_error("rk4 with the tree needs fss_tree_build on the same particle count");
        return FSS_ERR_STATE;
    }
    FSS_TRY(ctx->rk_k.ensure(sizeof(double) * 16 * n));
    FSS_TRY(ctx->rk_y.ensure(sizeof(double) * 4 * n));
    S = State{x, y, z, vort, area, false};
    if (!use_tree || T.p0 != T.n) return FSS_OK;
    FSS_TRY(ctx->rk_t.ensure(sizeof(double) * 5 * n));
    double *t = ctx->rk_t.as<double>();
    S = State{t, t + n, t + 2 * n, t + 3 * n, t + 4 * n, true};
    hipLaunchKernelGGL(k_rk4_load, dim3((unsigned)div_up(n, 256)), dim3(256), 0, ctx->stream, x, y, z, vort, area,
                       T.recid.as<int32_t>(), n, t);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

static fss_status finish(fss_ctx *ctx, const State &S, double *x, double *y, double *z, double *vort, int64_t n)
{
    if (!S.tree_order) return FSS_OK;
    hipLaunchKernelGGL(k_rk4_store, dim3((unsigned)div_up(n, 256)), dim3(256), 0, ctx->stream,
                       ctx->rk_t.as<double>(), ctx->tree.recid.as<int32_t>(), n, x, y, z, vort);
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

fss_status rk4_step(fss_ctx *ctx, double *x, double *y, double *z, double *vort, const double *area,
                    int64_t n, double dt, int use_tree)
{
    State S;
    FSS_TRY(begin(ctx, x, y, z, vort, area, n, use_tree, S));
    FSS_TRY(step(ctx, S, n, dt, use_tree));
    return finish(ctx, S, x, y, z, vort, n);
}

fss_status rk4_run_graph(fss_ctx *ctx, double *x, double *y, double *z, double *vort,
                         const double *area, int64_t n, double dt, int use_tree, int steps)
{
    if (steps <= 0) return FSS_OK;
    State S;
    FSS_TRY(begin(ctx, x, y, z, vort, area, n, use_tree, S));
    // the graph holds the addresses of the state and of the workspace and the
    // plan's launch shapes of its capture: any reallocation since then (a larger
    // direct sum on this context) or another near tile means capturing again; the
    // entries that build or tune a tree drop the graph themselves
    const void *key[6] = {S.x, S.y, S.z, S.vort, S.area, nullptr};
    bool same = ctx->graph_exec && ctx->graph_n == n && ctx->graph_dt == dt &&
                ctx->graph_tree == use_tree && ctx->graph_near_r == ctx->near_r &&
                ctx->graph_epoch == alloc_epoch();
    for (int i = 0; i < 5 && same; i++) same = ctx->graph_key[i] == key[i];
    int done = 0;
    if (!same) {
        if (ctx->graph_exec) {
            (void)hipGraphExecDestroy(ctx->graph_exec);
            ctx->graph_exec = nullptr;
        }
        if (ctx->graph) {
            (void)hipGraphDestroy(ctx->graph);
            ctx->graph = nullptr;
        }
        // eager first step sizes every workspace, so the capture allocates nothing
        FSS_TRY(step(ctx, S, n, dt, use_tree));
        done = 1;
        ctx->capturing = true;
        FSS_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        fss_status st = step(ctx, S, n, dt, use_tree);
        hipGraph_t gr = nullptr;
        hipError_t e = hipStreamEndCapture(ctx->stream, &gr);
        ctx->capturing = false;
        if (st != FSS_OK) {
            if (gr) (void)hipGraphDestroy(gr);
            return st;
        }
        FSS_HIP(e);
        ctx->graph = gr;
        FSS_HIP(hipGraphInstantiate(&ctx->graph_exec, gr, nullptr, nullptr, 0));
        for (int i = 0; i < 5; i++) ctx->graph_key[i] = key[i];
        ctx->graph_n = n;
        ctx->graph_dt = dt;
        ctx->graph_tree = use_tree;
        ctx->graph_near_r = ctx->near_r;
        ctx->graph_epoch = alloc_epoch();
    }
    for (int i = done; i < steps; i++) FSS_HIP(hipGraphLaunch(ctx->graph_exec, ctx->stream));
    return finish(ctx, S, x, y, z, vort, n);
}

} // namespace fss
