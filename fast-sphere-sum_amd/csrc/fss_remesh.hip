// fss_remesh.hip -- remesh onto the regular grid (regrid_points2
// remesh.h:109-178, tri_interp helpers.h:251-265).
//
// After an RK4 step the particles (the vertices of the Lagrangian mesh) have
// moved; every grid point (target) takes the absolute vorticity interpolated
// linearly on the advected triangle that contains it.  Search order as in the
// reference: the triangles adjacent to the target's own vertex first, in the
// given order, then every triangle in index order; the first triangle whose
// raw barycentric coordinates are all >= 0 (check_in_tri helpers.h:159-163)
// wins.
//
// Compiled with -ffp-contract=off: the barycentric solve (fss_geom.h, netlib
// order) decides the containing triangle and the interpolation is summed in
// the reference's order.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>

#include "fss_geom.h"
#include "fss_internal.h"

namespace fss {

namespace {

__device__ inline void load_tri(const int32_t *__restrict__ tris, int64_t t, const double *__restrict__ ax,
                                const double *__restrict__ ay, const double *__restrict__ az, int32_t *tv,
                                double *v)
{
    for (int m = 0; m < 3; m++) {
        tv[m] = tris[3 * t + m];
        v[3 * m] = ax[tv[m]];
        v[3 * m + 1] = ay[tv[m]];
        v[3 * m + 2] = az[tv[m]];
    }
}

__device__ inline bool in_tri(const double *v, const double *p, double *c)
{
    fssg::barycoords(v, v + 3, v + 6, p, c);
    return (c[0] >= 0) && (c[1] >= 0) && (c[2] >= 0);
}

// tri_interp: normalised coordinates (scaled by the reciprocal of their sum,
// norm_barycoords helpers.h:152-157), absolute vorticity interpolated, the
// relative vorticity recovered at the target; the tracer interpolated directly
__device__ inline void interp(const int32_t *tv, const double *c, const double *__restrict__ az,
                              const double *__restrict__ avort, const double *__restrict__ atr, double tz,
                              double omega, double *vort_out, double *tr_out)
{
    double r = 1.0 / (c[0] + c[1] + c[2]);
    double b0 = c[0] * r, b1 = c[1] * r, b2 = c[2] * r;
    double a0 = avort[tv[0]] + 2 * omega * az[tv[0]];
    double a1 = avort[tv[1]] + 2 * omega * az[tv[1]];
    double a2 = avort[tv[2]] + 2 * omega * az[tv[2]];
    double a = b0 * a0 + b1 * a1 + b2 * a2;
    *vort_out = a - 2 * omega * tz;
    if (atr) *tr_out = b0 * atr[tv[0]] + b1 * atr[tv[1]] + b2 * atr[tv[2]];
}

// False only where the solve cannot make p a non-negative combination of the
// vertices.  Its coordinates are exact for vertices perturbed by a small
// multiple of 1e-16 of the largest one (LU with pivoting is backward stable), and
// coordinate m times the determinant is p . (v_{m+1} x v_{m+2}): two of these
// with opposite signs beyond 1e-12 |p| max|v|^2 keep opposite signs under any such
// perturbation.  A matrix that could be singular under one (its solve stops at a
// zero pivot and leaves p in place of coordinates) and anything not finite are
// left to the solve.
__device__ inline bool may_hold(const double *v, const double *p)
{
    double f[3], vv = 0, det = 0;
    for (int m = 0; m < 3; m++) {
        const double *a = v + 3 * ((m + 1) % 3), *b = v + 3 * ((m + 2) % 3);
        const double c0 = a[1] * b[2] - a[2] * b[1], c1 = a[2] * b[0] - a[0] * b[2], c2 = a[0] * b[1] - a[1] * b[0];
        f[m] = p[0] * c0 + p[1] * c1 + p[2] * c2;
        vv = fmax(vv, a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
        if (m == 0) det = v[0] * c0 + v[1] * c1 + v[2] * c2;
    }
    const double tol = 1e-12 * vv * (fabs(p[0]) + fabs(p[1]) + fabs(p[2]));
    return !(det * det > 1e-24 * vv * vv * vv && fmin(f[0], fmin(f[1], f[2])) < -tol && fmax(f[0], fmax(f[1], f[2])) > tol);
}

// Adjacent triangles of the target's vertex; misses go to the fallback list.
// A target first walks to a triangle that may hold it and then solves, so the
// targets of a wave solve together and nearly always once (163,842 targets: 21.7
// us; solving every triangle on the way 24.3, eight lanes a target 25.9).
__global__ void __launch_bounds__(256) k_remesh_adjacent(
    int64_t n, const double *__restrict__ ax, const double *__restrict__ ay, const double *__restrict__ az,
    const double *__restrict__ avort, const double *__restrict__ atr, const int32_t *__restrict__ tris,
    const int32_t *__restrict__ vt_off, const int32_t *__restrict__ vt_idx, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, double omega, double *vort, double *tr,
    int32_t *tri_out, int32_t *miss, unsigned long long *nmiss)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double p[3] = {x[i], y[i], z[i]};
    double v[9], c[3];
    int32_t tv[3], t = -1;
    int32_t j = vt_off[i];
    const int32_t end = vt_off[i + 1];
    for (;;) {
        bool may = false;
        while (j < end && !may) {
            t = vt_idx[j++];
            load_tri(tris, t, ax, ay, az, tv, v);
            may = may_hold(v, p);
        }
        if (!may) break;
        if (in_tri(v, p, c)) {
            interp(tv, c, az, avort, atr, p[2], omega, &vort[i], tr ? &tr[i] : nullptr);
            tri_out[i] = t;
            return;
        }
    }
    tri_out[i] = -1;
    unsigned long long q = atomicAdd(nmiss, 1ull);
    miss[q] = (int32_t)i;
}

// ------------------------------------------------------------------
// full search of the missed targets: the lowest-index triangle of all that
// contains the target
// ------------------------------------------------------------------
// Scanning every triangle for every missed target is ntri solves each (5,472
// targets of 327,680 triangles: 16 ms).  A target in the cone of a triangle's
// vertices lies within the cap around their mean direction (any cap up to a
// hemisphere is convex), so the triangles are binned by the cell of that
// direction in a cubic grid over [-1, 1]^3, and a target solves only the
// triangles of the cells around it whose cap holds it.
//
// The solve rounds: a triangle also "contains" a target that rounding puts
// there.  With condition number k of the vertex matrix the coordinates are off
// by a small multiple of 1e-16 k relative to the largest, so below k = 1e6
// coordinates that come out non-negative are above -1e-8 of the largest one and the
// target is within 1.0000001 of the triangle's size of its centre: the caps are
// 1.05 times as large, and 2e-6 for their rounding to FP32.  Triangles that are worse conditioned, not finite, or
// larger than the cells (RM_CAP) stay on a list that every target solves.
struct RmGrid {
    int G;       // cells per dimension
    float inv;   // cells per unit length
    float rmax;  // largest chord radius that is binned
};

__device__ inline int rm_cell1(const RmGrid &g, float x)
{
    const int k = (int)((x + 1.0f) * g.inv);
    return k < 0 ? 0 : k < g.G ? k : g.G - 1;
}

// unit vector of p; false where there is none
__device__ inline bool rm_unit(const double *p, float *u)
{
    const double q = p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
    const float r = rsqrtf((float)q);
    for (int k = 0; k < 3; k++) u[k] = (float)p[k] * r;
    return q > 1e-30 && q < 1e30;
}

// Cap of a triangle in FP32: unit axis and the chord from it to the furthest
// vertex direction, each off by less than 1e-6 (the searches add that); false
// where the triangle is not to be binned.  The condition number is estimated
// from edge differences formed in FP64; the line is drawn at 1e6, where their
// FP32 products still tell.
__device__ inline bool rm_cap(const double *v, float *axis, float &chord)
{
    float u[9], s[3];
    bool ok = rm_unit(v, u) && rm_unit(v + 3, u + 3) && rm_unit(v + 6, u + 6);
    for (int k = 0; k < 3; k++) s[k] = u[k] + u[3 + k] + u[6 + k];
    const float q = s[0] * s[0] + s[1] * s[1] + s[2] * s[2], r = rsqrtf(q);
    float d2 = 0, e[9];
    for (int k = 0; k < 3; k++) axis[k] = s[k] * r;
    for (int m = 0; m < 3; m++) {
        float d = 0;
        for (int k = 0; k < 3; k++) {
            d += (u[3 * m + k] - axis[k]) * (u[3 * m + k] - axis[k]);
            e[3 * m + k] = (float)(v[(3 * m + 3 + k) % 9] - v[3 * m + k]);
        }
        d2 = fmaxf(d2, d);
    }
    chord = sqrtf(d2);
    // |v_j x v_k| <= |v| |edge|, det = v_0 . (e_0 x e_1)
    float len2 = 0, edge2 = 0;
    for (int m = 0; m < 3; m++) {
        const float w0 = (float)v[3 * m], w1 = (float)v[3 * m + 1], w2 = (float)v[3 * m + 2];
        len2 = fmaxf(len2, w0 * w0 + w1 * w1 + w2 * w2);
        edge2 = fmaxf(edge2, e[3 * m] * e[3 * m] + e[3 * m + 1] * e[3 * m + 1] + e[3 * m + 2] * e[3 * m + 2]);
    }
    const float det = (float)v[0] * (e[1] * e[5] - e[2] * e[4]) + (float)v[1] * (e[2] * e[3] - e[0] * e[5]) +
                      (float)v[2] * (e[0] * e[4] - e[1] * e[3]);
    return ok && q > 0.1f && 3.0f * len2 * sqrtf(edge2) < 1e6f * fabsf(det); // false for anything not finite
}

__global__ void __launch_bounds__(256) k_remesh_bin(int64_t ntri, const double *__restrict__ ax,
                                                    const double *__restrict__ ay, const double *__restrict__ az,
                                                    const int32_t *__restrict__ tris, RmGrid g, int32_t *count,
                                                    int2 *place, float4 *cap, int32_t *odd, unsigned int *nodd)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntri) return;
    int32_t tv[3];
    double v[9];
    float a[3], chord;
    load_tri(tris, t, ax, ay, az, tv, v);
    if (rm_cap(v, a, chord) && chord <= g.rmax) {
        const int c = (rm_cell1(g, a[2]) * g.G + rm_cell1(g, a[1])) * g.G + rm_cell1(g, a[0]);
        place[t] = make_int2(c, atomicAdd(&count[c], 1));
        cap[t] = make_float4(a[0], a[1], a[2], chord);
    } else {
        place[t] = make_int2(-1, 0);
        odd[atomicAdd(nodd, 1u)] = (int32_t)t;
    }
}

__global__ void __launch_bounds__(256) k_remesh_sort(int64_t ntri, const int2 *__restrict__ place,
                                                     const int32_t *__restrict__ start, int32_t *bin)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < ntri && place[t].x >= 0) bin[start[place[t].x] + place[t].y] = (int32_t)t;
}

// one wave per missed target
__global__ void __launch_bounds__(256) k_remesh_full(
    const int32_t *__restrict__ miss, int64_t nmiss, const double *__restrict__ ax, const double *__restrict__ ay,
    const double *__restrict__ az, const double *__restrict__ avort, const double *__restrict__ atr,
    const int32_t *__restrict__ tris, RmGrid g, const int32_t *__restrict__ start, const int32_t *__restrict__ bin,
    const float4 *__restrict__ cap, const int32_t *__restrict__ odd, const unsigned int *__restrict__ nodd,
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z, double omega,
    double *vort, double *tr, int32_t *tri_out, unsigned long long *nbad)
{
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= nmiss) return;
    const int lane = threadIdx.x & 63;
    const int64_t i = miss[w];
    const double p[3] = {x[i], y[i], z[i]};
    double v[9], c[3];
    float u[3];
    int32_t tv[3], best = INT32_MAX;
    auto test = [&](int32_t t) {
        if (t >= best) return;
        load_tri(tris, t, ax, ay, az, tv, v);
        if (may_hold(v, p) && in_tri(v, p, c)) best = t;
    };
    if (rm_unit(p, u)) {
        const float q = 1.05f * g.rmax + 4e-6f;
        int lo[3], hi[3];
        for (int k = 0; k < 3; k++) {
            lo[k] = rm_cell1(g, u[k] - q);
            hi[k] = rm_cell1(g, u[k] + q);
        }
        for (int cz = lo[2]; cz <= hi[2]; cz++)
            for (int cy = lo[1]; cy <= hi[1]; cy++) {
                // the cells of a row are consecutive, and so are their triangles
                const int32_t row = (cz * g.G + cy) * g.G;
                const int32_t e = start[row + hi[0] + 1];
                for (int32_t k = start[row + lo[0]] + lane; k < e; k += 64) {
                    const int32_t t = bin[k];
                    const float4 a = cap[t];
                    const float dx = u[0] - a.x, dy = u[1] - a.y, dz = u[2] - a.z, r = 1.05f * a.w + 2e-6f;
                    if (dx * dx + dy * dy + dz * dz <= r * r) test(t);
                }
            }
    } else {
        // no direction: such a target is in no cap
        for (int64_t t = lane; t < start[(int64_t)g.G * g.G * g.G]; t += 64) test(bin[t]);
    }
    for (unsigned k = lane; k < *nodd; k += 64) test(odd[k]);
    for (int o = 32; o > 0; o >>= 1) best = min(best, __shfl_xor(best, o, 64));
    if (lane != 0) return;
    if (best == INT32_MAX) {
        tri_out[i] = -1;
        atomicAdd(nbad, 1ull);
        return;
    }
    load_tri(tris, best, ax, ay, az, tv, v);
    in_tri(v, p, c);
    interp(tv, c, az, avort, atr, p[2], omega, &vort[i], tr ? &tr[i] : nullptr);
    tri_out[i] = best;
}

// Cells: a triangle of the mean size (4 pi / ntri, circumradius r0) may be four
// times larger and is still binned, a cell is two such radii wide (a target then
// looks at 8 cells at most, about 50 triangles each), at most 192 cells a side
// (28 MB of counts).
constexpr int RM_MAX_G = 192;
static RmGrid rm_grid(int64_t ntri)
{
    const double r0 = std::sqrt(4 * M_PI / (1.3 * (double)ntri)), rmax = std::min(0.5, 4 * r0);
    RmGrid g;
    g.G = (int)std::max(1.0, std::min((double)RM_MAX_G, std::floor(2.0 / (2.1 * rmax))));
    g.inv = g.G / 2.0f;
    g.rmax = (float)rmax;
    return g;
}

} // namespace

fss_status remesh(fss_ctx *ctx, const double *ax, const double *ay, const double *az, const double *avort,
                  const double *atr, const int32_t *tris, int64_t ntri, const int32_t *vt_off,
                  const int32_t *vt_idx, const double *x, const double *y, const double *z, double *vort,
                  double *tr, int32_t *tri_out, int64_t n, double omega, int64_t *n_fallback, int64_t *n_missing)
{
    hipStream_t s = ctx->stream;
    Remesh &W = ctx->remesh;
    // counters: [0] misses, [1] targets in no triangle, [2] triangles outside the bins
    FSS_TRY(W.cnt.ensure(sizeof(unsigned long long) * 3));
    FSS_TRY(W.miss.ensure(sizeof(int32_t) * n));
    int32_t *to = tri_out;
    if (!to) {
        FSS_TRY(W.tri.ensure(sizeof(int32_t) * n));
        to = W.tri.as<int32_t>();
    }
    FSS_HIP(hipMemsetAsync(W.cnt.p, 0, sizeof(unsigned long long) * 3, s));
    unsigned long long *c = W.cnt.as<unsigned long long>();
    int32_t *miss = W.miss.as<int32_t>();
    hipLaunchKernelGGL(k_remesh_adjacent, dim3((unsigned)div_up(n, 256)), dim3(256), 0, s, n, ax, ay, az, avort,
                       atr, tris, vt_off, vt_idx, x, y, z, omega, vort, tr, to, miss, c);
    FSS_HIP(hipGetLastError());
    unsigned long long h[2] = {0, 0};
    FSS_TRY(read_back(ctx, h, c, sizeof(unsigned long long)));
    if (h[0] > 0) {
        const RmGrid g = rm_grid(ntri);
        const int64_t nc = (int64_t)g.G * g.G * g.G;
        size_t tmp = 0;
        FSS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, (int32_t *)nullptr, (int32_t *)nullptr, (int)(nc + 1), s));
        FSS_TRY(W.count.ensure(sizeof(int32_t) * (nc + 1)));
        FSS_TRY(W.start.ensure(sizeof(int32_t) * (nc + 1)));
        FSS_TRY(W.scan.ensure(tmp));
        FSS_TRY(W.place.ensure(sizeof(int2) * ntri));
        FSS_TRY(W.cap.ensure(sizeof(float4) * ntri));
        FSS_TRY(W.bin.ensure(sizeof(int32_t) * ntri));
        FSS_TRY(W.odd.ensure(sizeof(int32_t) * ntri));
        unsigned int *nodd = reinterpret_cast<unsigned int *>(c + 2);
        const dim3 gt((unsigned)div_up(ntri, 256));
        FSS_HIP(hipMemsetAsync(W.count.p, 0, sizeof(int32_t) * (nc + 1), s));
        hipLaunchKernelGGL(k_remesh_bin, gt, dim3(256), 0, s, ntri, ax, ay, az, tris, g, W.count.as<int32_t>(),
                           W.place.as<int2>(), W.cap.as<float4>(), W.odd.as<int32_t>(), nodd);
        FSS_HIP(hipcub::DeviceScan::ExclusiveSum(W.scan.p, tmp, W.count.as<int32_t>(), W.start.as<int32_t>(),
                                                 (int)(nc + 1), s));
        hipLaunchKernelGGL(k_remesh_sort, gt, dim3(256), 0, s, ntri, W.place.as<int2>(), W.start.as<int32_t>(),
                           W.bin.as<int32_t>());
        hipLaunchKernelGGL(k_remesh_full, dim3((unsigned)div_up((int64_t)h[0], 4)), dim3(256), 0, s, miss, (int64_t)h[0],
                           ax, ay, az, avort, atr, tris, g, W.start.as<int32_t>(), W.bin.as<int32_t>(),
                           W.cap.as<float4>(), W.odd.as<int32_t>(), nodd, x, y, z, omega, vort, tr, to, c + 1);
        FSS_HIP(hipGetLastError());
        FSS_TRY(read_back(ctx, h + 1, c + 1, sizeof(unsigned long long)));
    }
    if (n_fallback) *n_fallback = (int64_t)h[0];
    if (n_missing) *n_missing = (int64_t)h[1];
    if (h[1] > 0) return set_error("remesh: a target lies in no triangle of the advected mesh"), FSS_ERR_NUMERIC;
    return FSS_OK;
}

} // namespace fss
