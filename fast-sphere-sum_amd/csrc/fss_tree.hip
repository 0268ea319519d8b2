// fss_tree.hip -- icosahedral tree, point location, node lists, dual
// traversal and evaluation plan, all built on the device.
//
// Compiled with -ffp-contract=off: the geometry and the 3x3 solves decide
// integer tree data and must round exactly as the reference's operation
// order does (see fss_geom.h).
//
// Reference map (Old-BVE-code/):
//   icos_init            icos_utils.h:15-133   -> k_geom_level0, k_geom_children
//   points_assign        icos_utils.h:145-190  -> k_locate
//   tree_tri_points      icos_utils.h:165      -> ranges of the records in tree order; the
//                                                 lists themselves on export only
//   tree_traverse        fast_rhs.h:16-91      -> k_trav_classify / k_trav_scatter
//     The reference pops a FIFO queue and appends the 4 children of a split
//     pair at its tail.  FIFO order processes the queue generation by
//     generation (every pair of generation g is popped before any pair of
//     generation g+1), and inside a generation in the order the pairs were
//     appended.  Each generation is therefore one data-parallel pass:
//     classify every pair, add up the emitted and the split pairs before it,
//     scatter.  Emitted pairs land in the list in exactly the reference's
//     order.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>

#include "fss_geom.h"
#include "fss_internal.h"

namespace fss {

using fssg::level_offset;
using fssg::level_size;

// ------------------------------------------------------------------
// geometry
// ------------------------------------------------------------------
__global__ void k_geom_level0(double *tri_xyz, double *tri_info, double radius)
{
    int i = threadIdx.x;
    if (i >= 20) return;
    fssg::IcosBase b;
    fssg::icos_base(&b);
    double v[3][3];
    for (int m = 0; m < 3; m++) fssg::project_to_sphere_2(b.v[b.f[i][m] - 1], radius, v[m]);
    for (int m = 0; m < 3; m++)
        for (int k = 0; k < 3; k++) tri_xyz[9 * i + 3 * m + k] = v[m][k];
    double c[3];
    fssg::tri_center(v[0], v[1], v[2], radius, c);
    double r = fssg::tri_radius(v[0], v[1], v[2], c);
    tri_info[4 * i + 0] = c[0];
    tri_info[4 * i + 1] = c[1];
    tri_info[4 * i + 2] = c[2];
    tri_info[4 * i + 3] = r;
}

__global__ void k_geom_children(double *tri_xyz, double *tri_info, int64_t parent_off,
                                int64_t child_off, int64_t nparent, double radius)
{
    int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nparent) return;
    const double *P = tri_xyz + 9 * (parent_off + j);
    double v1[3], v2[3], v3[3];
    for (int k = 0; k < 3; k++) {
        v1[k] = P[k];
        v2[k] = P[3 + k];
        v3[k] = P[6 + k];
    }
    double v12[3], v23[3], v31[3];
    fssg::midpoints(v1, v2, v3, radius, v12, v23, v31);
    for (int c = 0; c < 4; c++) {
        const double *tv[3], *cv[3];
        fssg::child_tri(c, v1, v2, v3, v12, v23, v31, tv, cv);
        int64_t g = child_off + 4 * j + c;
        for (int m = 0; m < 3; m++)
            for (int k = 0; k < 3; k++) tri_xyz[9 * g + 3 * m + k] = tv[m][k];
        double ce[3];
        fssg::tri_center(cv[0], cv[1], cv[2], radius, ce);
        double r = fssg::tri_radius(cv[0], cv[1], cv[2], ce);
        tri_info[4 * g + 0] = ce[0];
        tri_info[4 * g + 1] = ce[1];
        tri_info[4 * g + 2] = ce[2];
        tri_info[4 * g + 3] = r;
    }
}

// inverse of the vertex matrix [v1 v2 v3] of every node: row m is
// (v_{m+1} x v_{m+2}) / det, so that the barycentric coordinates of p are
// c_m = row_m . p
__global__ void k_tinv(const double *__restrict__ tri_xyz, int64_t nn, double *tinv)
{
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nn) return;
    const double *T = tri_xyz + 9 * g;
    double r[3][3];
    for (int m = 0; m < 3; m++) {
        const double *a = T + 3 * ((m + 1) % 3), *b = T + 3 * ((m + 2) % 3);
        r[m][0] = a[1] * b[2] - a[2] * b[1];
        r[m][1] = a[2] * b[0] - a[0] * b[2];
        r[m][2] = a[0] * b[1] - a[1] * b[0];
    }
    double det = T[0] * r[0][0] + T[1] * r[0][1] + T[2] * r[0][2];
    double id = 1.0 / det;
    for (int m = 0; m < 3; m++)
        for (int k = 0; k < 3; k++) tinv[9 * g + 3 * m + k] = r[m][k] * id;
}

// per triangle: norm of its centre and arc radius of its cap
__global__ void k_geo_aux(const double *__restrict__ tri_info, int64_t nt, double2 *aux)
{
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nt) return;
    const double *ti = tri_info + 4 * g;
    aux[g] = make_double2(fssg::norm3(ti), 2.0 * asin(0.5 * ti[3]));
}

// ------------------------------------------------------------------
// point location (icos_utils.h:145-170)
// ------------------------------------------------------------------
// What a build counts on the device, read back at its three synchronisations.
struct BuildInfo {
    unsigned long long nexc;        // exception memberships
    unsigned long long dropped[13]; // particles on no list, per level
    unsigned long long margin;      // bits of min |separation - theta|
    long long nF[28], nE[28];       // pairs of a generation; interactions emitted before it
    long long needF, needI;         // capacities that would have held the traversal
    int overflow;
    unsigned long long types[4];
    unsigned long long pairs[3]; // near and far evaluations, entries of the near source lists
    int4 totals;                 // near items, interpolant slots, near output slots, charge nodes
    int4 up;                     // upward items of <= 32 records, longer ones, nodes with several, partials
    int n_proxy;
};

// A particle takes the first child whose solved coordinates are all >= 0.
// Solving every child on the way was most of the kernel (200,003 particles, 6
// levels: 143 us); the rows of the inverse vertex matrix tell a child that
// cannot pass from nine products.  The solve's coordinates are exact for
// vertices moved by a few 1e-15, which moves coordinate m times the determinant
// by that times |p|; the determinant of a level-l triangle is above 0.28 / 4^l, so
// below -8e-12 4^l |p| a coordinate is negative in the solve too.  The lanes of a
// wave walk to their next candidate and solve together.
// The key of the main path is formed on the way: it holds one digit per level,
// the level-0 node (0..19, 20 = not found), then the child digit (0..3) while
// covered, 4 after the path ends.
template <typename Key>
__global__ void __launch_bounds__(256) k_locate(const double *__restrict__ x, const double *__restrict__ y,
                                                const double *__restrict__ z, int64_t n, int L,
                                                const double *__restrict__ tri_xyz,
                                                const double *__restrict__ tinv, int robust, int32_t *loc,
                                                uint8_t *found, Key *keys, int32_t *vals, int32_t *ecnt,
                                                BuildInfo *info)
{
    int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const double p[3] = {x[id], y[id], z[id]};
    double tol = 8e-12 * (fabs(p[0]) + fabs(p[1]) + fabs(p[2]));
    int prev = 0;
    bool cov = true;
    Key key = 0;
    for (int l = 0; l < L; l++, tol *= 4) {
        const int lb = l > 0 ? 4 * prev : 0, ub = l > 0 ? lb + 4 : 20;
        const int64_t lo = level_offset(l);
        int hit = -1, j = lb;
        for (;;) {
            bool may = false;
            while (j < ub && !may) {
                const double *R = tinv + 9 * (lo + j++);
                const double c0 = R[0] * p[0] + R[1] * p[1] + R[2] * p[2];
                const double c1 = R[3] * p[0] + R[4] * p[1] + R[5] * p[2];
                const double c2 = R[6] * p[0] + R[7] * p[1] + R[8] * p[2];
                may = !(c0 < -tol || c1 < -tol || c2 < -tol);
            }
            if (!may) break;
            const double *T = tri_xyz + 9 * (lo + j - 1);
            double c[3];
            fssg::barycoords(T, T + 3, T + 6, p, c);
            if ((c[0] >= 0) && (c[1] >= 0) && (c[2] >= 0)) {
                hit = j - 1;
                break;
            }
        }
        if (hit < 0 && robust) {
            // none passes (points on edges): the largest minimum coordinate
            hit = lb;
            double bestmin = -INFINITY;
            for (j = lb; j < ub; j++) {
                const double *T = tri_xyz + 9 * (lo + j);
                double c[3];
                fssg::barycoords(T, T + 3, T + 6, p, c);
                double mn = c[0] < c[1] ? c[0] : c[1];
                mn = mn < c[2] ? mn : c[2];
                if (mn > bestmin) {
                    bestmin = mn;
                    hit = j;
                }
            }
        }
        // a particle that passes no child keeps location 0 (icos_utils.h:139-140)
        const int lc = hit >= 0 ? hit : 0;
        const bool f = hit >= 0;
        loc[(int64_t)l * n + id] = lc;
        found[(int64_t)l * n + id] = f ? 1 : 0;
        cov = cov && f;
        const int digit = l == 0 ? (cov ? lc : 20) : (cov ? lc - 4 * prev : 4);
        key = l == 0 ? (Key)digit : key * 5 + (Key)digit;
        if (!f) atomicAdd(&info->dropped[l], 1ull); // rare
        if (!cov && f) {                            // exception membership (rare)
            atomicAdd(&ecnt[lo + lc], 1);
            atomicAdd(&info->nexc, 1ull);
        }
        prev = lc;
    }
    keys[id] = key;
    vals[id] = (int32_t)id;
}

// ------------------------------------------------------------------
// tree order of the source records
// ------------------------------------------------------------------
struct Pow5 {
    unsigned long long v[13]; // 5^(L-1-l)
};

// Main range of every node, record node (deepest node of the main path) and
// particle of every main record, from the sorted keys alone: a node's range
// starts and ends where the key's leading digits change.
template <typename Key>
__global__ void __launch_bounds__(256) k_main_ranges(const Key *__restrict__ keys, const int32_t *__restrict__ perm,
                                                     const uint8_t *__restrict__ found, int64_t n, int L, Pow5 pw,
                                                     int4 *nrange, int32_t *recid, int32_t *recnode, uint8_t *rinfo,
                                                     int32_t *ipos)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Key k = keys[i];
    const Key kp = i > 0 ? keys[i - 1] : 0, kn = i + 1 < n ? keys[i + 1] : 0;
    int32_t deepest = 0, idx = 0;
    int e = 0; // levels on the main path
    Key rem = k;
    for (int l = 0; l < L; l++) {
        const Key w = (Key)pw.v[l], d = rem / w;
        if (d >= (Key)(l == 0 ? 20 : 4)) break;
        rem -= d * w;
        idx = l == 0 ? (int32_t)d : 4 * idx + (int32_t)d;
        const int64_t g = level_offset(l) + idx;
        const Key pk = k / w;
        if (i == 0 || kp / w != pk) nrange[g].x = (int32_t)i;
        if (i == n - 1 || kn / w != pk) nrange[g].y = (int32_t)(i + 1);
        deepest = (int32_t)g;
        e = l + 1;
    }
    const int32_t id = perm[i];
    bool exc = false;
    for (int l = e + 1; l < L; l++) exc = exc || found[(int64_t)l * n + id];
    recid[i] = id;
    recnode[i] = deepest;
    rinfo[i] = (uint8_t)(e | (exc ? 0x80 : 0));
    ipos[id] = (int32_t)i;
}

__global__ void k_level_keys(const int32_t *loc, const uint8_t *found, int64_t n, uint32_t sentinel,
                             uint32_t *keys, int32_t *vals)
{
    int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    bool f = found[id] != 0;
    keys[id] = f ? (uint32_t)loc[id] : sentinel;
    vals[id] = (int32_t)id;
}

// exception memberships: (node, particle) of every level a particle is on a
// list outside its main path
__global__ void k_exc_fill(const int32_t *__restrict__ loc, const uint8_t *__restrict__ found, int64_t n,
                           int L, unsigned long long *counter, unsigned long long *keys, int32_t *vals)
{
    int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    bool cov = true;
    for (int l = 0; l < L; l++) {
        bool f = found[(int64_t)l * n + id] != 0;
        cov = cov && f;
        if (!cov && f) {
            unsigned long long q = atomicAdd(counter, 1ull);
            int64_t g = level_offset(l) + loc[(int64_t)l * n + id];
            keys[q] = ((unsigned long long)g << 32) | (unsigned long long)id;
            vals[q] = (int32_t)id;
        }
    }
}

__global__ void k_exc_ranges(const unsigned long long *__restrict__ keys, const int32_t *__restrict__ vals,
                             int64_t ne, int64_t base, int4 *nrange, int32_t *recid, int32_t *recnode)
{
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ne) return;
    int64_t g = (int64_t)(keys[q] >> 32);
    if (q == 0 || (int64_t)(keys[q - 1] >> 32) != g) nrange[g].z = (int32_t)(base + q);
    recid[base + q] = vals[q];
    recnode[base + q] = (int32_t)g;
}

// main members (nrange holds start and end until here), list length
__global__ void k_nrange_counts(const int32_t *__restrict__ ecnt, int64_t nn, int4 *nrange, int32_t *counts)
{
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nn) return;
    int4 r = nrange[g];
    r.y -= r.x;
    r.w = ecnt[g];
    nrange[g] = r;
    counts[g] = r.y + r.w;
}

// ------------------------------------------------------------------
// traversal (fast_rhs.h:16-91)
// ------------------------------------------------------------------
// A generation is two launches of TRAV_BLOCKS blocks, each on one contiguous
// chunk of the generation's pairs: classify leaves the chunk's numbers of
// emitted and split pairs, scatter adds up those of the chunks before its own
// and writes its pairs in order.  The sizes of the generations stay on the
// device, so all of them are launched without waiting for one (the host read
// four numbers back per generation: 11 generations, about 4 of a 13 ms build);
// what does not fit the buffers is counted and not written, and the host starts
// again with larger ones.
constexpr int TRAV_BLOCKS = 512;

enum : int8_t { ACT_SKIP = -1, ACT_SPLIT_T = 4, ACT_SPLIT_S = 5 };

__global__ void k_trav_init(int4 *F, BuildInfo *info)
{
    int i = threadIdx.x + blockIdx.x * blockDim.x;
    if (i == 0) {
        info->nF[0] = 400;
        info->margin = (unsigned long long)__double_as_longlong(INFINITY);
    }
    if (i >= 400) return;
    F[i] = make_int4(i / 20, i % 20, 0, 0);
}

// separation (r_t + r_s) / distance of the MAC (fast_rhs.h:37-41); a pair
// within FSS_MAC_TIE of theta is decided with the correctly rounded distance,
// so the list does not depend on the last bit of the device's acos.  aux: the
// norms of the centres.
__device__ inline void mac_separation(const double *ti, const double *si, double nt, double ns, double radius,
                                      double theta, double &distance, double &separation)
{
    double cl = fssg::dot3(ti, si) / (nt * ns); // great_circ_dist
    if (cl < -1.0) cl = -1.0;
    if (1.0 < cl) cl = 1.0;
    distance = acos(cl) * radius;
    separation = (ti[3] + si[3]) / distance;
    if (distance > 0 && fabs(separation - theta) <= FSS_MAC_TIE) {
        distance = fssg::great_circ_dist_cr(ti, si, radius);
        separation = (ti[3] + si[3]) / distance;
    }
}

// The MAC's theta per level of a pair's coarser node: theta at the leaf
// level, times theta_decay per level towards the root (repeated products
// from the leaves up, so host code forms the same doubles).
struct MacTheta {
    double t[13];
};
static MacTheta mac_thetas(int L, double theta, double decay)
{
    MacTheta m{};
    m.t[L - 1] = theta;
    for (int l = L - 2; l >= 0; l--) m.t[l] = m.t[l + 1] * decay;
    return m;
}

// BLTC admits a pair only if the two nodes' caps are apart: the MAC compares
// chord radii with the arc distance of the centres, so at theta near 1 it
// admits triangles that share a vertex (their caps touch there), whose
// corner proxies coincide and whose kernel is singular.  The caps' arc
// radii 2 asin(r/2) (geo_aux) must sum to less than the distance, with a relative
// margin of 1e-12 that settles exact touching (centres and the shared vertex
// on one great circle) the same way on every machine.  Below theta 0.98 at
// every level this never removes a pair: the largest node (level 0) has
// r = 0.641 and 2 asin(r/2) <= 1.02 r there, so the arc radii sum to less
// than 1.02 x 0.98 d.
__device__ inline bool caps_apart(double at, double as, double distance)
{
    return at + as < distance * (1.0 - 1e-12);
}

__device__ inline int64_t trav_chunk(int64_t nF) { return 256 * ((nF + 256 * TRAV_BLOCKS - 1) / (256 * TRAV_BLOCKS)); }

__global__ void __launch_bounds__(256) k_trav_classify(const int4 *__restrict__ F, BuildInfo *info, int gen,
                                                       const int32_t *__restrict__ counts,
                                                       const double *__restrict__ tri_info,
                                                       const double2 *__restrict__ aux, MacTheta thetas,
                                                       int many_count, int L, double radius, int bltc, int8_t *act,
                                                       int2 *blk, int4 *types)
{
    const int64_t nF = info->nF[gen], chunk = trav_chunk(nF), base = (int64_t)blockIdx.x * chunk;
    if (nF == 0) return;
    if (base >= nF) {
        if (threadIdx.x == 0) blk[blockIdx.x] = make_int2(0, 0);
        return;
    }
    unsigned long long mb = ~0ull;
    int ne = 0, ns = 0, ty[4] = {0, 0, 0, 0};
    for (int64_t i = base + threadIdx.x; i < min(base + chunk, nF); i += 256) {
        const int4 q = F[i];
        const int ct = q.x, cs = q.y, lt = q.z, ls = q.w;
        const double theta = thetas.t[min(lt, ls)];
        const int64_t gt = level_offset(lt) + ct, gs = level_offset(ls) + cs;
        const int32_t nt = counts[gt], nsrc = counts[gs];
        int8_t a = ACT_SKIP;
        if (nt != 0 && nsrc != 0) {
            const double2 at = aux[gt], as = aux[gs];
            double distance, separation;
            mac_separation(tri_info + 4 * gt, tri_info + 4 * gs, at.x, as.x, radius, theta, distance, separation);
            if (distance > 0) {
                const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(separation - theta));
                mb = b < mb ? b : mb;
            }
            if ((distance > 0) && (separation < theta) && (!bltc || caps_apart(at.y, as.y, distance))) {
                a = (int8_t)((nt > many_count ? 2 : 0) + (nsrc > many_count ? 1 : 0));
            } else if ((nt < many_count) && (nsrc < many_count)) {
                a = 0;
            } else if ((lt == L - 1) && (ls == L - 1)) {
                a = 0;
            } else if (lt == L - 1) {
                a = ACT_SPLIT_S;
            } else if (ls == L - 1) {
                a = ACT_SPLIT_T;
            } else if (nt >= nsrc) {
                a = ACT_SPLIT_T;
            } else {
                a = ACT_SPLIT_S;
            }
        }
        act[i] = a;
        ne += (a >= 0 && a <= 3) ? 1 : 0;
        ns += (a == ACT_SPLIT_T || a == ACT_SPLIT_S) ? 1 : 0;
#pragma unroll
        for (int t = 0; t < 4; t++) ty[t] += a == t ? 1 : 0;
    }
    __shared__ int red[4][6];
    __shared__ unsigned long long mred[4];
    int v[6] = {ne, ns, ty[0], ty[1], ty[2], ty[3]};
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int k = 0; k < 6; k++) v[k] += __shfl_xor(v[k], o, 64);
        const unsigned long long m = __shfl_xor(mb, o, 64);
        mb = m < mb ? m : mb;
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        for (int k = 0; k < 6; k++) red[wave][k] = v[k];
        mred[wave] = mb;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < 4; w++) {
        for (int k = 0; k < 6; k++) red[0][k] += red[w][k];
        mb = mred[w] < mb ? mred[w] : mb;
    }
    blk[blockIdx.x] = make_int2(red[0][0], red[0][1]);
    // every block keeps its own type counts over the generations
    int4 tt = types[blockIdx.x];
    tt.x += red[0][2];
    tt.y += red[0][3];
    tt.z += red[0][4];
    tt.w += red[0][5];
    types[blockIdx.x] = tt;
    if (mb < *(volatile unsigned long long *)&info->margin) atomicMin(&info->margin, mb);
}

__global__ void __launch_bounds__(256) k_trav_scatter(const int4 *__restrict__ F, BuildInfo *info, int gen,
                                                      const int8_t *__restrict__ act, const int2 *__restrict__ blk,
                                                      const int32_t *__restrict__ counts, int32_t *inter,
                                                      int64_t capI, int4 *Fn, int64_t capF)
{
    const int64_t nF = info->nF[gen], chunk = trav_chunk(nF), base = (int64_t)blockIdx.x * chunk;
    const bool last = blockIdx.x == TRAV_BLOCKS - 1; // also writes the next generation's sizes
    if (nF == 0 || (base >= nF && !last)) return;
    __shared__ long long pre[4][2];
    __shared__ int wtot[4][2];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    long long e = 0, sp = 0;
    for (int j = threadIdx.x; j < (int)blockIdx.x; j += 256) {
        const int2 b = blk[j];
        e += b.x;
        sp += b.y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        e += __shfl_xor(e, o, 64);
        sp += __shfl_xor(sp, o, 64);
    }
    if (lane == 0) {
        pre[wave][0] = e;
        pre[wave][1] = sp;
    }
    __syncthreads();
    long long E = info->nE[gen], S = 0;
    for (int w = 0; w < 4; w++) {
        E += pre[w][0];
        S += pre[w][1];
    }
    for (int64_t b = base; b < min(base + chunk, nF); b += 256) {
        const int64_t i = b + threadIdx.x;
        const int8_t a = i < nF ? act[i] : (int8_t)ACT_SKIP;
        const bool em = a >= 0 && a <= 3, spl = a == ACT_SPLIT_T || a == ACT_SPLIT_S;
        const uint64_t me = __ballot(em), ms = __ballot(spl), below = ((uint64_t)1 << lane) - 1;
        __syncthreads();
        if (lane == 0) {
            wtot[wave][0] = __popcll(me);
            wtot[wave][1] = __popcll(ms);
        }
        __syncthreads();
        long long pe = E + __popcll(me & below), ps = S + __popcll(ms & below);
        for (int w = 0; w < 4; w++) {
            if (w < wave) {
                pe += wtot[w][0];
                ps += wtot[w][1];
            }
            E += wtot[w][0];
            S += wtot[w][1];
        }
        if (em && pe < capI) {
            const int4 q = F[i];
            int32_t *o = inter + 7 * pe;
            o[0] = q.z;
            o[1] = q.w;
            o[2] = q.x;
            o[3] = q.y;
            o[4] = counts[level_offset(q.z) + q.x];
            o[5] = counts[level_offset(q.w) + q.y];
            o[6] = a;
        } else if (spl && 4 * ps + 4 <= capF) {
            const int4 q = F[i];
            int4 *d = Fn + 4 * ps;
            for (int c = 0; c < 4; c++)
                d[c] = a == ACT_SPLIT_T ? make_int4(4 * q.x + c, q.y, q.z + 1, q.w)
                                        : make_int4(q.x, 4 * q.y + c, q.z, q.w + 1);
        }
    }
    if (!last || threadIdx.x != 0) return;
    info->nE[gen + 1] = E;
    if (E > capI || 4 * S > capF) {
        info->overflow = 1;
        if (E > info->needI) info->needI = E;
        if (4 * S > info->needF) info->needF = 4 * S;
    }
    info->nF[gen + 1] = 4 * S > capF ? 0 : 4 * S; // a generation cut short ends the traversal
}

// number of interactions of each type (pp, pc, cp, cc)
__global__ void __launch_bounds__(TRAV_BLOCKS) k_trav_types(const int4 *__restrict__ types, BuildInfo *info)
{
    __shared__ int4 s[TRAV_BLOCKS];
    s[threadIdx.x] = types[threadIdx.x];
    __syncthreads();
    if (threadIdx.x >= 4) return;
    unsigned long long t = 0;
    for (int b = 0; b < TRAV_BLOCKS; b++) t += (unsigned)(&s[b].x)[threadIdx.x];
    info->types[threadIdx.x] = t;
}

// Proxy items: the class-B ranges of every interpolant slot cut into parts of
// about `chunk` sources, in range order (a part closes at the range
// that takes its count to the chunk size, or at the slot's last range).  One
// wave per slot, counting first and writing after the scan of the counts; a
// slot with fewer sources than the chunk size in all is one part.
__device__ inline int32_t chunk_parts(const ProxyItem &it, const Range *__restrict__ rb, int chunk, ProxyItem *out,
                                      int32_t slot)
{
    int32_t np = 0, b = it.b_beg;
    int64_t acc = 0;
    for (int32_t r = it.b_beg; r < it.b_end; r++) {
        acc += rb[r].count & ~FSS_SELF_BIT;
        if (acc >= chunk || r + 1 == it.b_end) {
            if (out) out[np] = ProxyItem{it.node, b, r + 1, slot};
            np++;
            b = r + 1;
            acc = 0;
        }
    }
    return np;
}

// Sources per part: FSS_PROXY_CHUNK, or so many that a small tree's parts are 1.5
// for each SIMD (a wave takes a part, and the longest ends the kernel): FP64 fast
// sum as the reference has it, N = 10,242, one context alone, 53.7 us with parts of
// 4,096, 43.1 of 2,048, 38.9 of 1,024, 38.4 of 512; trees of 30,000 particles and more
// have the items anyway.  Mixed precision keeps 4,096, since the parts' starts
// decide which FP32 values share a partial sum; so do a batch's instances, which
// fill the chip together.
static int proxy_chunk(const fss_ctx *ctx)
{
    if (ctx->cfg.precision == FSS_MIXED || ctx->batch_part) return FSS_PROXY_CHUNK;
    const int64_t c = 128 * div_up(ctx->tree.n_far_src, 128 * 1536);
    return (int)std::min<int64_t>(FSS_PROXY_CHUNK, std::max<int64_t>(512, c));
}

// sources of the slot (all lanes hold the sum)
__device__ inline int64_t slot_sources(const ProxyItem &it, const Range *__restrict__ rb)
{
    long long c = 0;
    for (int r = it.b_beg + (int)(threadIdx.x & 63); r < it.b_end; r += 64) c += rb[r].count & ~FSS_SELF_BIT;
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    return c;
}

__global__ void __launch_bounds__(256) k_chunk_count(const ProxyItem *__restrict__ one, int64_t nslot,
                                                     const Range *__restrict__ rb, int chunk, int32_t *cnt)
{
    const int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (q >= nslot) return;
    const ProxyItem it = one[q];
    const bool split = slot_sources(it, rb) >= chunk;
    if ((threadIdx.x & 63) == 0) cnt[q] = split ? chunk_parts(it, rb, chunk, nullptr, (int32_t)q) : it.b_end > it.b_beg ? 1 : 0;
}

__global__ void __launch_bounds__(256) k_chunk_fill(const ProxyItem *__restrict__ one, int64_t nslot,
                                                    const Range *__restrict__ rb, const int32_t *__restrict__ pos,
                                                    int chunk, ProxyItem *parts, ProxySlot *slots, BuildInfo *info)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nslot) return;
    const int32_t p0 = pos[q], np = pos[q + 1] - p0;
    const ProxyItem it = one[q];
    if (np == 1) parts[p0] = ProxyItem{it.node, it.b_beg, it.b_end, (int32_t)q};
    else chunk_parts(it, rb, chunk, parts + p0, (int32_t)q);
    slots[q] = ProxySlot{it.node, p0, p0 + np, 0};
    if (q == nslot - 1) info->n_proxy = pos[nslot];
}

// ------------------------------------------------------------------
// evaluation plan
// ------------------------------------------------------------------
// class of an interaction: 0 = direct targets (A), 1 = proxy targets (B).
// PARITY (rhs_eval.h:34-45): pp, pc -> A with particle sources; cp, cc -> B
// with particle sources.  BLTC: pp -> A particles, pc -> A proxies,
// cp -> B particles, cc -> B proxies.
__global__ void k_plan_keys(const int32_t *__restrict__ inter, int64_t m, uint32_t nn,
                            uint32_t *keys, int32_t *vals)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int32_t *o = inter + 7 * i;
    const uint32_t cls = (o[6] == 0 || o[6] == 1) ? 0u : 1u;
    keys[i] = cls * nn + (uint32_t)(level_offset(o[0]) + o[2]);
    vals[i] = (int32_t)i;
}

// ranges per sorted interaction: 1, or 2 for particle sources whose node has
// exception members (main range + exception range); only needed where such
// members exist
__global__ void k_plan_rcount(const int32_t *__restrict__ inter, const int32_t *__restrict__ sorted_idx,
                              int64_t m, const int4 *__restrict__ nrange, int bltc, int32_t *nr)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k > m) return;
    if (k == m) {
        nr[k] = 0;
        return;
    }
    const int32_t *o = inter + 7 * (int64_t)sorted_idx[k];
    int type = o[6];
    int64_t gs = level_offset(o[1]) + o[3];
    bool proxy_src = bltc && (type == 1 || type == 3);
    nr[k] = (!proxy_src && nrange[gs].w > 0) ? 2 : 1;
}

// Source ranges of every interaction in sorted order (rpos: position of each,
// null = its own index), class A to ra, class B (from nA on) to rb; flags the
// charge nodes (BLTC: sources of pc and cc).  Grid-stride: the evaluation counts
// are summed per block and added once (an atomic per wave of 28,000 waves had
// been most of the kernel: 344 us for 1.8 M interactions).
__global__ void __launch_bounds__(256) k_plan_ranges(const int32_t *__restrict__ inter,
                                                     const int32_t *__restrict__ sorted_idx,
                                                     const uint32_t *__restrict__ sorted_keys,
                                                     const int32_t *__restrict__ rpos, int64_t m, int64_t nA,
                                                     const int4 *__restrict__ nrange, int bltc, int p, int64_t p0,
                                                     Range *ra, Range *rb, uint32_t *rkeys, uint8_t *charge,
                                                     BuildInfo *info)
{
    unsigned long long acc[3] = {0, 0, 0};
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < m; k += (int64_t)gridDim.x * 256) {
        const int32_t *o = inter + 7 * (int64_t)sorted_idx[k];
        const int lt = o[0], ls = o[1], ct = o[2], cs = o[3], type = o[6];
        const int64_t gs = level_offset(ls) + cs;
        const bool proxy_src = bltc && (type == 1 || type == 3), clsA = type == 0 || type == 1;
        const unsigned long long srcn = proxy_src ? (unsigned long long)p : (unsigned long long)o[5];
        if (clsA) {
            const int4 t = nrange[level_offset(lt) + ct];
            acc[0] += (unsigned long long)o[4] * srcn;
            acc[2] += (unsigned long long)((t.y + 63) / 64 + (t.w + 63) / 64) * srcn;
        } else {
            acc[1] += (unsigned long long)p * srcn;
        }
        const int64_t q = rpos ? rpos[k] : k;
        Range *out = q < nA ? ra + q : rb + (q - nA);
        Range r;
        r.node = (int32_t)gs;
        r.pad = 0;
        if (rkeys) rkeys[q] = sorted_keys[k];
        if (proxy_src) {
            r.start = (int32_t)(p0 + gs * p);
            r.count = p;
            out[0] = r;
            charge[gs] = 1;
            continue;
        }
        // particle sources of a node that contains the target node: the self
        // pair may lie in these ranges
        const int self = (clsA && ls <= lt && (ct >> (2 * (lt - ls))) == cs) ? FSS_SELF_BIT : 0;
        const int4 nr = nrange[gs];
        r.start = nr.x;
        r.count = nr.y | self;
        out[0] = r;
        if (nr.w > 0) {
            r.start = nr.z;
            r.count = nr.w | self;
            out[1] = r;
            rkeys[q + 1] = sorted_keys[k];
        }
    }
    __shared__ unsigned long long red[4][3];
    for (int c = 0; c < 3; c++) {
        for (int o = 32; o > 0; o >>= 1) acc[c] += __shfl_xor(acc[c], o, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = acc[c];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int c = threadIdx.x;
        const unsigned long long t = red[0][c] + red[1][c] + red[2][c] + red[3][c];
        if (t) atomicAdd(&info->pairs[c], t);
    }
}

__global__ void k_plan_segments(const uint32_t *__restrict__ keys, int64_t m, uint32_t nn,
                                int32_t *beg, int32_t *end)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    uint32_t key = keys[k];
    if (k == 0 || keys[k - 1] != key) beg[key] = (int32_t)k;
    if (k == m - 1 || keys[k + 1] != key) end[key] = (int32_t)(k + 1);
}

// per node (and a zero after the last): near chunks (main and exception
// targets), proxy work, output slots of its targets, modified charges
__global__ void k_plan_nodes(const int32_t *__restrict__ beg, const int32_t *__restrict__ end,
                             const int4 *__restrict__ nrange, const uint8_t *__restrict__ charge, uint32_t nn,
                             int4 *per)
{
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g > nn) return;
    if (g == nn) {
        per[g] = make_int4(0, 0, 0, 0);
        return;
    }
    const bool a = end[g] > beg[g], b = end[nn + g] > beg[nn + g];
    const int4 r = nrange[g];
    per[g] = make_int4(a ? (int32_t)((r.y + 63) / 64 + (r.w + 63) / 64) : 0, b ? 1 : 0, a ? r.y + r.w : 0, charge[g]);
}

struct Add4 {
    __host__ __device__ int4 operator()(const int4 &a, const int4 &b) const
    {
        return make_int4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
    }
};

// pos: exclusive scan of k_plan_nodes
__global__ void k_plan_items(const int32_t *__restrict__ beg, const int32_t *__restrict__ end,
                             const int4 *__restrict__ nrange, const int4 *__restrict__ pos, uint32_t nn, int64_t nA,
                             NearItem *near, ProxyItem *prox, int32_t *node_slot, int32_t *oslot, int32_t *charge)
{
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nn) return;
    const int4 at = pos[g], nx = pos[g + 1];
    node_slot[g] = nx.y > at.y ? at.y : -1;
    oslot[g] = nx.z > at.z ? at.z : -1;
    if (nx.w > at.w) charge[at.w] = (int32_t)g;
    if (nx.y > at.y) {
        ProxyItem it;
        it.node = (int32_t)g;
        it.b_beg = (int32_t)(beg[nn + g] - nA);
        it.b_end = (int32_t)(end[nn + g] - nA);
        it.slot = at.y;
        prox[at.y] = it;
    }
    if (nx.x == at.x) return;
    int4 r = nrange[g];
    int32_t item = at.x, ob = at.z;
    for (int part = 0; part < 2; part++) {
        int32_t c = part ? r.w : r.y, off = part ? r.z : r.x;
        for (int32_t q = 0; 64 * q < c; q++) {
            NearItem it;
            it.tgt_start = off + 64 * q;
            it.tgt_cnt = min(64, c - 64 * q);
            it.a_beg = beg[g];
            it.a_end = end[g];
            it.node = (int32_t)g;
            it.out_base = ob + 64 * q;
            near[item++] = it;
        }
        ob += c;
    }
}

// node of every particle per level (-1 where the particle is not on a list)
__global__ void k_plan_nodeof(const int32_t *__restrict__ loc, const uint8_t *__restrict__ found,
                              int L, int64_t n, int32_t *nodeof)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)L * n) return;
    int l = (int)(i / n);
    nodeof[i] = found[i] ? (int32_t)(level_offset(l) + loc[i]) : -1;
}

// inverse map for the final per-particle reduction: the output slot of every
// near target, per level (one 64-thread block per near item)
__global__ void k_plan_inverse(const NearItem *__restrict__ items, const int32_t *__restrict__ recid, int L,
                               int64_t n, int32_t *inv_active)
{
    const NearItem it = items[blockIdx.x];
    int t = threadIdx.x;
    if (t >= it.tgt_cnt) return;
    int lev = 0;
    while (lev + 1 < L && level_offset(lev + 1) <= it.node) lev++;
    inv_active[(int64_t)lev * n + recid[it.tgt_start + t]] = it.out_base + t;
}

// static proxy positions of every node: planar u v1 + v v2 + (1-u-v) v3
// (fast_rhs.h:188-200) in PARITY, its projection onto the sphere in BLTC.
__global__ void k_proxy_xyz(const double *__restrict__ tri_xyz, const double *__restrict__ pts,
                            int p, int64_t nn, int spherical, double4 *proxy)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nn * p) return;
    int64_t g = i / p;
    int k = (int)(i % p);
    const double *T = tri_xyz + 9 * g;
    double u = pts[3 * k], v = pts[3 * k + 1];
    double q[3];
    if (!spherical) {
        for (int c = 0; c < 3; c++) {
            double p1 = T[c] * u, p2 = T[3 + c] * v, p3 = T[6 + c] * (1.0 - u - v);
            q[c] = (p1 + p2) + p3;
        }
    } else {
        double w = pts[3 * k + 2];
        for (int c = 0; c < 3; c++) q[c] = u * T[c] + v * T[3 + c] + w * T[6 + c];
        double r = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
        for (int c = 0; c < 3; c++) q[c] /= r;
    }
    proxy[i] = make_double4(q[0], q[1], q[2], 0.0);
}

// ------------------------------------------------------------------
// host orchestration
// ------------------------------------------------------------------
static int bits_for64(uint64_t maxkey)
{
    int b = 1;
    while (b < 64 && ((uint64_t)1 << b) <= maxkey) b++;
    return b;
}

template <typename Key>
static fss_status cub_sort_pairs(DevBuf &tmp, const Key *kin, Key *kout, const int32_t *vin, int32_t *vout, int64_t n,
                                 int bits, hipStream_t s)
{
    size_t bytes = 0;
    FSS_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, kin, kout, vin, vout, (int)n, 0, bits, s));
    FSS_TRY(tmp.ensure(bytes));
    FSS_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, kin, kout, vin, vout, (int)n, 0, bits, s));
    return FSS_OK;
}

template <typename T> static fss_status cub_exclusive_sum(DevBuf &tmp, const T *in, T *out, int64_t n, hipStream_t s)
{
    size_t bytes = 0;
    FSS_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, s));
    FSS_TRY(tmp.ensure(bytes));
    FSS_HIP(hipcub::DeviceScan::ExclusiveSum(tmp.p, bytes, in, out, (int)n, s));
    return FSS_OK;
}

static fss_status cub_exclusive_add4(DevBuf &tmp, const int4 *in, int4 *out, int64_t n, hipStream_t s)
{
    size_t bytes = 0;
    const int4 zero = make_int4(0, 0, 0, 0);
    FSS_HIP(hipcub::DeviceScan::ExclusiveScan(nullptr, bytes, in, out, Add4(), zero, (int)n, s));
    FSS_TRY(tmp.ensure(bytes));
    FSS_HIP(hipcub::DeviceScan::ExclusiveScan(tmp.p, bytes, in, out, Add4(), zero, (int)n, s));
    return FSS_OK;
}

// The build's arrays that start at zero, in one buffer cleared by one memset (six
// of them took 3 us each of the host)
struct ZeroParts {
    size_t types, ecnt, begend, charge, bytes; // after the BuildInfo
    explicit ZeroParts(int64_t nn)
    {
        types = (sizeof(BuildInfo) + 15) / 16 * 16;
        ecnt = types + sizeof(int4) * TRAV_BLOCKS;
        begend = ecnt + sizeof(int32_t) * nn;
        charge = begend + sizeof(int32_t) * 4 * nn;
        bytes = charge + nn;
    }
};

// The build's scratch arrays stay with the context while they are small
// (allocating and freeing about forty of them was 5 of a 13 ms build) and are
// given back after a build that needed more than this.
constexpr size_t BUILD_SCRATCH_KEEP = (size_t)256 << 20;

void build_scratch_trim(BuildScratch &B)
{
    size_t total = 0;
    for (DevBuf *b : B.all()) total += b->bytes;
    if (total > BUILD_SCRATCH_KEEP)
        for (DevBuf *b : B.all()) b->release();
}

// Triangles of levels 0 .. levels-1: fixed by the depth alone (the sphere has
// radius 1), and the triangles of a shallower tree are the first ones of a
// deeper, so a context computes them once for its deepest tree.  Matrices and caps
// are of the nodes, which end a level earlier (on all levels they were 88 bytes a
// triangle in place of 22: 1.85 GB at 10 levels).
static fss_status geo_ensure(fss_ctx *ctx, int levels)
{
    Geo &G = ctx->geo;
    hipStream_t s = ctx->stream;
    if (G.levels >= levels) return FSS_OK;
    G.levels = 0;
    const int64_t nt = level_offset(levels), nn = level_offset(levels - 1);
    FSS_TRY(G.xyz.ensure(sizeof(double) * 9 * nt));
    FSS_TRY(G.info.ensure(sizeof(double) * 4 * nt));
    FSS_TRY(G.tinv.ensure(sizeof(double) * 9 * nn));
    FSS_TRY(G.aux.ensure(sizeof(double2) * nn));
    const double radius = ctx->cfg.radius;
    hipLaunchKernelGGL(k_geom_level0, dim3(1), dim3(64), 0, s, G.xyz.as<double>(), G.info.as<double>(), radius);
    for (int l = 0; l + 1 < levels; l++) {
        const int64_t np = level_size(l);
        hipLaunchKernelGGL(k_geom_children, dim3((unsigned)div_up(np, 256)), dim3(256), 0, s, G.xyz.as<double>(),
                           G.info.as<double>(), level_offset(l), level_offset(l + 1), np, radius);
    }
    hipLaunchKernelGGL(k_tinv, dim3((unsigned)div_up(nn, 256)), dim3(256), 0, s, G.xyz.as<double>(), nn,
                       G.tinv.as<double>());
    hipLaunchKernelGGL(k_geo_aux, dim3((unsigned)div_up(nn, 256)), dim3(256), 0, s, G.info.as<double>(), nn,
                       G.aux.as<double2>());
    FSS_HIP(hipGetLastError());
    G.levels = levels;
    return FSS_OK;
}

// point location and tree order of the main records (keys of type Key)
template <typename Key>
static fss_status locate_and_sort(fss_ctx *ctx, const double *x, const double *y, const double *z, int64_t n,
                                  uint64_t maxkey, const Pow5 &pw, int32_t *ecnt)
{
    Tree &T = ctx->tree;
    BuildScratch &B = ctx->build;
    hipStream_t s = ctx->stream;
    const unsigned gp = (unsigned)div_up(n, 256);
    FSS_TRY(B.k0.ensure(sizeof(Key) * n));
    FSS_TRY(B.k1.ensure(sizeof(Key) * n));
    FSS_TRY(B.v0.ensure(sizeof(int32_t) * n));
    FSS_TRY(B.v1.ensure(sizeof(int32_t) * n));
    hipLaunchKernelGGL((k_locate<Key>), dim3(gp), dim3(256), 0, s, x, y, z, n, T.L, T.d_xyz, T.d_tinv,
                       ctx->cfg.assign_mode == FSS_ASSIGN_ROBUST ? 1 : 0, T.loc.as<int32_t>(), T.found.as<uint8_t>(),
                       B.k0.as<Key>(), B.v0.as<int32_t>(), ecnt, B.info.as<BuildInfo>());
    FSS_TRY(cub_sort_pairs(B.cub, B.k0.as<Key>(), B.k1.as<Key>(), B.v0.as<int32_t>(), B.v1.as<int32_t>(), n,
                           bits_for64(maxkey), s));
    hipLaunchKernelGGL((k_main_ranges<Key>), dim3(gp), dim3(256), 0, s, B.k1.as<Key>(), B.v1.as<int32_t>(),
                       T.found.as<uint8_t>(), n, T.L, pw, T.nrange.as<int4>(), T.recid.as<int32_t>(),
                       T.recnode.as<int32_t>(), T.rinfo.as<uint8_t>(), T.ipos.as<int32_t>());
    FSS_HIP(hipGetLastError());
    return FSS_OK;
}

static fss_status too_many(int64_t ninter)
{
    // the plan indexes interactions and their source ranges (at most two per
    // interaction) with int32
    set_error("tree_build: " + std::to_string(ninter) + " interactions exceed the plan's 32-bit indices (at most " +
              std::to_string(INT32_MAX / 2) + "); use fewer tree levels or a larger theta");
    return FSS_ERR_INVALID;
}

fss_status tree_build(fss_ctx *ctx, const double *x, const double *y, const double *z, int64_t n)
{
    const fss_config &cfg = ctx->cfg;
    hipStream_t s = ctx->stream;
    Tree &T = ctx->tree;
    BuildScratch &B = ctx->build;
    const int L = cfg.tree_levels;
    const int p = ctx->interp.p;
    const bool bltc = cfg.eval_mode == FSS_EVAL_BLTC;
    if (L < 1 || L > 13) {
        set_error("tree_levels must be in [1, 13]");
        return FSS_ERR_INVALID;
    }
    if (n < 1 || n > (int64_t)INT32_MAX || (int64_t)L * n > (int64_t)INT32_MAX) {
        set_error("particle count out of range for 32-bit list offsets");
        return FSS_ERR_INVALID;
    }
    T.built = false;
    T.L = L;
    T.n = n;
    T.nn = level_offset(L);
    T.ntri_all = level_offset(L + 1);
    const uint32_t nn = (uint32_t)T.nn;
    const unsigned gn = (unsigned)div_up(T.nn + 1, 256);
    T.stats = fss_tree_stats{};
    T.stats.n = n;
    T.stats.tree_levels = L;
    T.stats.n_nodes = T.nn;
    T.ninst = 1;
    T.batched = false;

    // ---- geometry: levels 0..L (icos_init builds tree_levels refinements) ----
    FSS_TRY(geo_ensure(ctx, L + 1));
    T.d_xyz = ctx->geo.xyz.as<double>();
    T.d_info = ctx->geo.info.as<double>();
    T.d_tinv = ctx->geo.tinv.as<double>();

    // ---- point location, tree order of the source records, list lengths ----
    const ZeroParts Z(T.nn);
    FSS_TRY(B.info.ensure(Z.bytes));
    FSS_TRY(T.loc.ensure(sizeof(int32_t) * L * n));
    FSS_TRY(T.found.ensure((size_t)L * n));
    FSS_TRY(T.counts.ensure(sizeof(int32_t) * T.nn));
    FSS_TRY(T.nrange.ensure(sizeof(int4) * T.nn));
    FSS_TRY(T.recid.ensure(sizeof(int32_t) * n));
    FSS_TRY(T.recnode.ensure(sizeof(int32_t) * n));
    FSS_TRY(T.rinfo.ensure(n));
    FSS_TRY(T.ipos.ensure(sizeof(int32_t) * n));
    BuildInfo *info = B.info.as<BuildInfo>();
    char *const zero = B.info.as<char>();
    int4 *const types = reinterpret_cast<int4 *>(zero + Z.types);
    int32_t *const ecnt = reinterpret_cast<int32_t *>(zero + Z.ecnt);
    int32_t *const beg = reinterpret_cast<int32_t *>(zero + Z.begend), *const end = beg + 2 * T.nn;
    uint8_t *const charge = reinterpret_cast<uint8_t *>(zero + Z.charge);
    FSS_HIP(hipMemsetAsync(zero, 0, Z.bytes, s));
    FSS_HIP(hipMemsetAsync(T.nrange.p, 0, sizeof(int4) * T.nn, s));
    uint64_t maxkey = 21;
    Pow5 pw{};
    pw.v[L - 1] = 1;
    for (int l = L - 2; l >= 0; l--) pw.v[l] = 5 * pw.v[l + 1];
    for (int l = 1; l < L; l++) maxkey *= 5;
    const bool key32 = maxkey <= UINT32_MAX;
    auto sorted_records = [&]() -> fss_status {
        return key32 ? locate_and_sort<uint32_t>(ctx, x, y, z, n, maxkey, pw, ecnt)
                     : locate_and_sort<unsigned long long>(ctx, x, y, z, n, maxkey, pw, ecnt);
    };
    FSS_TRY(sorted_records());
    hipLaunchKernelGGL(k_nrange_counts, dim3((unsigned)div_up(T.nn, 256)), dim3(256), 0, s, ecnt, T.nn,
                       T.nrange.as<int4>(), T.counts.as<int32_t>());

    // ---- traversal ----
    // Capacities: what an earlier build on this context held, at least an
    // estimate of the interactions from the acceptance criterion (about 30 / theta^2
    // per occupied node with one theta, twice that with a tightened one), and never
    // more than there can be: a pair of occupied nodes comes up once, to be
    // emitted or split in four.
    BuildInfo h;
    {
        const double occupied = (double)std::min<int64_t>(T.nn, (int64_t)L * n);
        const double est = std::min(60.0 / (cfg.theta * cfg.theta) * occupied, 4.0 * occupied * occupied);
        int64_t cap = (int64_t)std::min(est, 16777216.0);
        cap = std::max<int64_t>(cap, 1 << 16);
        int64_t capI = std::max<int64_t>(cap, (int64_t)(T.inter.bytes / (7 * sizeof(int32_t))));
        int64_t capF = std::max<int64_t>(cap, (int64_t)(B.f0.bytes / sizeof(int4)));
        const int gens = 2 * L - 1; // every split takes one of the pair's two nodes a level down
        FSS_TRY(B.blk.ensure(sizeof(int2) * TRAV_BLOCKS));
        for (;;) {
            FSS_TRY(B.f0.ensure(sizeof(int4) * capF));
            FSS_TRY(B.f1.ensure(sizeof(int4) * capF));
            FSS_TRY(B.act.ensure(capF));
            FSS_TRY(T.inter.ensure(sizeof(int32_t) * 7 * capI));
            hipLaunchKernelGGL(k_trav_init, dim3(2), dim3(256), 0, s, B.f0.as<int4>(), info);
            int4 *F = B.f0.as<int4>(), *Fn = B.f1.as<int4>();
            for (int g = 0; g < gens; g++) {
                hipLaunchKernelGGL(k_trav_classify, dim3(TRAV_BLOCKS), dim3(256), 0, s, F, info, g,
                                   T.counts.as<int32_t>(), T.d_info, ctx->geo.aux.as<double2>(),
                                   mac_thetas(L, cfg.theta, cfg.theta_decay), cfg.many_count, L, cfg.radius,
                                   bltc ? 1 : 0, B.act.as<int8_t>(), B.blk.as<int2>(), types);
                hipLaunchKernelGGL(k_trav_scatter, dim3(TRAV_BLOCKS), dim3(256), 0, s, F, info, g,
                                   B.act.as<int8_t>(), B.blk.as<int2>(), T.counts.as<int32_t>(),
                                   T.inter.as<int32_t>(), capI, Fn, capF);
                std::swap(F, Fn);
            }
            hipLaunchKernelGGL(k_trav_types, dim3(1), dim3(TRAV_BLOCKS), 0, s, types, info);
            FSS_HIP(hipGetLastError());
            FSS_TRY(read_back(ctx, &h, info, sizeof(h)));
            if (!h.overflow) break;
            if ((int64_t)h.needI > INT32_MAX / 2) return too_many((int64_t)h.needI);
            if ((int64_t)h.needF > INT32_MAX) return too_many((int64_t)h.needF);
            if ((int64_t)h.needI > capI) capI = std::max<int64_t>(2 * capI, (int64_t)h.needI);
            if ((int64_t)h.needF > capF) capF = std::max<int64_t>(2 * capF, (int64_t)h.needF);
            // sizes of the generations and the overflow marks start again
            FSS_HIP(hipMemsetAsync(info->nF, 0, offsetof(BuildInfo, types) - offsetof(BuildInfo, nF), s));
            FSS_HIP(hipMemsetAsync(types, 0, sizeof(int4) * TRAV_BLOCKS, s));
        }
    }
    const int64_t ninter = (int64_t)*std::max_element(h.nE, h.nE + 28);
    if (ninter > INT32_MAX / 2) return too_many(ninter);
    T.ngen = 0;
    while (T.ngen < 28 && h.nF[T.ngen] > 0) T.ngen++;
    T.ninter = ninter;
    std::memcpy(&T.stats.mac_margin, &h.margin, 8);
    T.stats.n_interactions = ninter;
    T.stats.n_generations = T.ngen;
    for (int t = 0; t < 4; t++) T.stats.n_type[t] = (int64_t)h.types[t];
    T.nlist = 0;
    for (int l = 0; l < L; l++) {
        T.stats.dropped[l] = (int64_t)h.dropped[l];
        T.nlist += n - T.stats.dropped[l];
    }

    // ---- exception records ----
    const int64_t ne = (int64_t)h.nexc;
    T.p0 = n + ne;
    if (T.p0 + T.nn * p > INT32_MAX) return set_error("tree: source records exceed 32-bit positions"), FSS_ERR_INVALID;
    if (ne > 0) {
        // the record arrays grow: the main records are written again
        FSS_TRY(T.recid.ensure(sizeof(int32_t) * T.p0));
        FSS_TRY(T.recnode.ensure(sizeof(int32_t) * T.p0));
        FSS_TRY(T.rinfo.ensure(T.p0));
        FSS_HIP(hipMemsetAsync(T.rinfo.p, 0, T.p0, s));
        FSS_HIP(hipMemsetAsync(T.nrange.p, 0, sizeof(int4) * T.nn, s));
        FSS_HIP(hipMemsetAsync(ecnt, 0, sizeof(int32_t) * T.nn, s));
        FSS_TRY(sorted_records());
        hipLaunchKernelGGL(k_nrange_counts, dim3((unsigned)div_up(T.nn, 256)), dim3(256), 0, s, ecnt,
                           T.nn, T.nrange.as<int4>(), T.counts.as<int32_t>());
        // exception memberships, sorted by (node, particle)
        using u64 = unsigned long long;
        const unsigned gp = (unsigned)div_up(n, 256);
        FSS_TRY(B.ek0.ensure(sizeof(u64) * ne));
        FSS_TRY(B.ek1.ensure(sizeof(u64) * ne));
        FSS_TRY(B.ev0.ensure(sizeof(int32_t) * ne));
        FSS_TRY(B.ev1.ensure(sizeof(int32_t) * ne));
        FSS_HIP(hipMemsetAsync(&info->nexc, 0, sizeof(u64), s));
        hipLaunchKernelGGL(k_exc_fill, dim3(gp), dim3(256), 0, s, T.loc.as<int32_t>(), T.found.as<uint8_t>(), n, L,
                           &info->nexc, B.ek0.as<u64>(), B.ev0.as<int32_t>());
        FSS_TRY(cub_sort_pairs(B.cub, B.ek0.as<u64>(), B.ek1.as<u64>(), B.ev0.as<int32_t>(), B.ev1.as<int32_t>(), ne,
                               32 + bits_for64((uint64_t)T.nn), s));
        hipLaunchKernelGGL(k_exc_ranges, dim3((unsigned)div_up(ne, 256)), dim3(256), 0, s, B.ek1.as<u64>(),
                           B.ev1.as<int32_t>(), ne, n, T.nrange.as<int4>(), T.recid.as<int32_t>(),
                           T.recnode.as<int32_t>());
        FSS_HIP(hipGetLastError());
    }

    // ---- evaluation plan ----
    FSS_TRY(T.proxy_xyz.ensure(sizeof(double4) * T.nn * p));
    hipLaunchKernelGGL(k_proxy_xyz, dim3((unsigned)div_up(T.nn * p, 256)), dim3(256), 0, s, T.d_xyz,
                       ctx->d_pts.as<double>(), p, T.nn, bltc ? 1 : 0, T.proxy_xyz.as<double4>());
    const int64_t m = ninter;
    const int64_t mA = T.stats.n_type[0] + T.stats.n_type[1]; // class-A interactions (sorted first)
    FSS_TRY(B.per.ensure(sizeof(int4) * (T.nn + 1)));
    FSS_TRY(B.pos.ensure(sizeof(int4) * (T.nn + 1)));
    int64_t nA = mA, nR = m; // ranges: one per interaction, two where a particle source node has exception members
    if (m > 0) {
        const unsigned gb = (unsigned)div_up(m, 256);
        FSS_TRY(B.keys.ensure(sizeof(uint32_t) * m));
        FSS_TRY(B.keys2.ensure(sizeof(uint32_t) * m));
        FSS_TRY(B.vals.ensure(sizeof(int32_t) * m));
        FSS_TRY(B.vals2.ensure(sizeof(int32_t) * m));
        hipLaunchKernelGGL(k_plan_keys, dim3(gb), dim3(256), 0, s, T.inter.as<int32_t>(), m, nn,
                           B.keys.as<uint32_t>(), B.vals.as<int32_t>());
        FSS_TRY(cub_sort_pairs(B.cub, B.keys.as<uint32_t>(), B.keys2.as<uint32_t>(), B.vals.as<int32_t>(),
                               B.vals2.as<int32_t>(), m, bits_for64(2ull * nn), s));
        uint32_t *rkeys = nullptr;
        int32_t *rpos = nullptr;
        if (ne > 0) {
            FSS_TRY(B.rcnt.ensure(sizeof(int32_t) * (m + 1)));
            FSS_TRY(B.rpos.ensure(sizeof(int32_t) * (m + 1)));
            rpos = B.rpos.as<int32_t>();
            hipLaunchKernelGGL(k_plan_rcount, dim3((unsigned)div_up(m + 1, 256)), dim3(256), 0, s,
                               T.inter.as<int32_t>(), B.vals2.as<int32_t>(), m, T.nrange.as<int4>(), bltc ? 1 : 0,
                               B.rcnt.as<int32_t>());
            FSS_TRY(cub_exclusive_sum(B.cub, B.rcnt.as<int32_t>(), rpos, m + 1, s));
            int32_t a = 0, r = 0;
            FSS_TRY(read_back(ctx, &a, rpos + mA, 4));
            FSS_TRY(read_back(ctx, &r, rpos + m, 4));
            nA = a;
            nR = r;
            FSS_TRY(B.rkeys.ensure(sizeof(uint32_t) * nR));
            rkeys = B.rkeys.as<uint32_t>();
        }
        FSS_TRY(T.ranges_a.ensure(sizeof(Range) * std::max<int64_t>(1, nA)));
        FSS_TRY(T.ranges_b.ensure(sizeof(Range) * std::max<int64_t>(1, nR - nA)));
        hipLaunchKernelGGL(k_plan_ranges, dim3((unsigned)std::min<int64_t>(gb, 512)), dim3(256), 0, s,
                           T.inter.as<int32_t>(), B.vals2.as<int32_t>(), B.keys2.as<uint32_t>(), rpos, m, nA,
                           T.nrange.as<int4>(), bltc ? 1 : 0, p, T.p0, T.ranges_a.as<Range>(), T.ranges_b.as<Range>(),
                           rkeys, charge, info);
        hipLaunchKernelGGL(k_plan_segments, dim3((unsigned)div_up(nR, 256)), dim3(256), 0, s,
                           rkeys ? rkeys : B.keys2.as<uint32_t>(), nR, nn, beg, end);
    } else {
        FSS_TRY(T.ranges_a.ensure(sizeof(Range)));
        FSS_TRY(T.ranges_b.ensure(sizeof(Range)));
    }
    T.n_ra = nA;
    T.n_rb = nR - nA;
    hipLaunchKernelGGL(k_plan_nodes, dim3(gn), dim3(256), 0, s, beg, end, T.nrange.as<int4>(),
                       charge, nn, B.per.as<int4>());
    FSS_TRY(cub_exclusive_add4(B.cub, B.per.as<int4>(), B.pos.as<int4>(), T.nn + 1, s));
    FSS_HIP(hipMemcpyAsync(&info->totals, B.pos.as<int4>() + T.nn, sizeof(int4), hipMemcpyDeviceToDevice, s));
    FSS_TRY(read_back(ctx, &h, info, sizeof(h)));
    T.pairs_near = T.stats.pairs_near = (int64_t)h.pairs[0];
    T.pairs_far = T.stats.pairs_far = (int64_t)h.pairs[1];
    T.n_near_src = (int64_t)h.pairs[2];
    T.n_far_src = (int64_t)h.pairs[1] / p;
    T.n_near = h.totals.x;
    T.n_slot = h.totals.y;
    T.nslot_out = h.totals.z;
    T.n_charge = h.totals.w;
    FSS_TRY(T.oslot.ensure(sizeof(int32_t) * T.nn));
    FSS_TRY(T.node_slot.ensure(sizeof(int32_t) * T.nn));
    FSS_TRY(T.near_items.ensure(sizeof(NearItem) * std::max<int64_t>(1, T.n_near)));
    FSS_TRY(T.charge_nodes.ensure(sizeof(int32_t) * std::max<int64_t>(1, T.n_charge)));
    FSS_TRY(B.prox_one.ensure(sizeof(ProxyItem) * std::max<int64_t>(1, T.n_slot)));
    hipLaunchKernelGGL(k_plan_items, dim3(gn), dim3(256), 0, s, beg, end, T.nrange.as<int4>(), B.pos.as<int4>(), nn,
                       nA, T.near_items.as<NearItem>(), B.prox_one.as<ProxyItem>(), T.node_slot.as<int32_t>(),
                       T.oslot.as<int32_t>(), T.charge_nodes.as<int32_t>());
    // Long class-B lists split into chunks of about `chunk` sources
    // (order inside a node is kept).  Every chunk but a slot's last holds that
    // many, so this many items are room enough; their number stays on the
    // device until the build's last synchronisation.
    const int chunk = proxy_chunk(ctx);
    const int64_t proxy_room = T.n_slot + T.n_far_src / chunk;
    FSS_TRY(T.proxy_slots.ensure(sizeof(ProxySlot) * std::max<int64_t>(1, T.n_slot)));
    FSS_TRY(T.proxy_items.ensure(sizeof(ProxyItem) * std::max<int64_t>(1, proxy_room)));
    if (T.n_slot > 0) {
        FSS_TRY(B.rcnt.ensure(sizeof(int32_t) * (T.n_slot + 1)));
        FSS_TRY(B.rpos.ensure(sizeof(int32_t) * (T.n_slot + 1)));
        FSS_HIP(hipMemsetAsync(B.rcnt.as<int32_t>() + T.n_slot, 0, sizeof(int32_t), s));
        hipLaunchKernelGGL(k_chunk_count, dim3((unsigned)div_up(T.n_slot, 4)), dim3(256), 0, s,
                           B.prox_one.as<ProxyItem>(), T.n_slot, T.ranges_b.as<Range>(), chunk, B.rcnt.as<int32_t>());
        FSS_TRY(cub_exclusive_sum(B.cub, B.rcnt.as<int32_t>(), B.rpos.as<int32_t>(), T.n_slot + 1, s));
        hipLaunchKernelGGL(k_chunk_fill, dim3((unsigned)div_up(T.n_slot, 256)), dim3(256), 0, s,
                           B.prox_one.as<ProxyItem>(), T.n_slot, T.ranges_b.as<Range>(), B.rpos.as<int32_t>(),
                           chunk, T.proxy_items.as<ProxyItem>(), T.proxy_slots.as<ProxySlot>(), info);
    }
    T.n_proxy = proxy_room;
    // maps of the memberships outside the main paths
    if (ne > 0) {
        FSS_TRY(T.nodeof.ensure(sizeof(int32_t) * (size_t)L * n));
        hipLaunchKernelGGL(k_plan_nodeof, dim3((unsigned)div_up((int64_t)L * n, 256)), dim3(256), 0, s,
                           T.loc.as<int32_t>(), T.found.as<uint8_t>(), L, n, T.nodeof.as<int32_t>());
        FSS_TRY(T.inv_active.ensure(sizeof(int32_t) * (size_t)L * n));
        FSS_HIP(hipMemsetAsync(T.inv_active.p, 0xff, sizeof(int32_t) * (size_t)L * n, s));
        if (T.n_near > 0)
            hipLaunchKernelGGL(k_plan_inverse, dim3((unsigned)T.n_near), dim3(64), 0, s, T.near_items.as<NearItem>(),
                               T.recid.as<int32_t>(), L, n, T.inv_active.as<int32_t>());
    }
    const Instance one{0, n, 0, L, 0, 0, 0};
    FSS_TRY(T.inst.ensure(sizeof(Instance)));
    FSS_HIP(hipMemcpyAsync(T.inst.p, &one, sizeof(Instance), hipMemcpyHostToDevice, s));
    FSS_HIP(hipGetLastError());
    if (ctx->batch_part) {
        // the merged plan is finished by the caller, who needs the item count;
        // without its source lists this one serves no evaluation, so it is not
        // built, should a later instance be refused
        FSS_TRY(read_back(ctx, &h, info, sizeof(h)));
        T.n_proxy = h.n_proxy;
        return FSS_OK;
    }
    FSS_TRY(plan_finish(ctx));
    build_scratch_trim(B);
    T.built = true;
    return FSS_OK;
}

// Source list of every near item: the records of its class-A ranges, the
// ranges that cannot hold one of the item's targets first, then the self
// ranges.  One wave per item.
__global__ void __launch_bounds__(64) k_near_src_count(NearItem *items, const Range *__restrict__ ranges,
                                                       int64_t *cnt)
{
    const int lane = threadIdx.x;
    NearItem it = items[blockIdx.x];
    int c0 = 0, c1 = 0;
    for (int r = it.a_beg + lane; r < it.a_end; r += 64) {
        const int32_t c = ranges[r].count;
        if (c & FSS_SELF_BIT) c1 += c & ~FSS_SELF_BIT;
        else c0 += c;
    }
    for (int off = 32; off > 0; off >>= 1) {
        c0 += __shfl_xor(c0, off, 64);
        c1 += __shfl_xor(c1, off, 64);
    }
    if (lane == 0) {
        items[blockIdx.x].n_other = c0;
        items[blockIdx.x].n_self = c1;
        cnt[blockIdx.x] = (int64_t)c0 + c1;
    }
}

// Writes the record positions of the ranges [beg, end) that `take` accepts (it
// is given a range's count) to dst, one wave together; returns the end of the
// list.  The lanes load 64 ranges at once and sum their counts; sixteen lanes
// then write a range, four ranges at a time (ranges hold a leaf, or up to 45
// proxies).  Range by range, every turn waited for its own load and wrote with ten
// lanes: 200,003 particles, theta 0.6: near lists 61 us, far lists 31; now 29 and
// 14 (level-10 grid, degree 7: 739 and 235, now 420 and 168).
template <typename Take>
__device__ inline int32_t *list_ranges(const Range *__restrict__ ranges, int beg, int end, int32_t *dst, Take take)
{
    const int lane = threadIdx.x & 63;
    for (int b = beg; b < end; b += 64) {
        int32_t start = 0, count = 0;
        if (b + lane < end) {
            const Range r = ranges[b + lane];
            start = r.start;
            count = take(r.count) ? r.count & ~FSS_SELF_BIT : 0;
        }
        int32_t sum = count;
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t t = __shfl_up(sum, o, 64);
            sum += lane >= o ? t : 0;
        }
        for (int l0 = 0; l0 < min(64, end - b); l0 += 4) {
            const int l = l0 + (lane >> 4);
            const int32_t s = __shfl(start, l, 64), c = __shfl(count, l, 64), o = __shfl(sum, l, 64) - c;
            for (int i = lane & 15; i < c; i += 16) dst[o + i] = s + i;
        }
        dst += __shfl(sum, 63, 64);
    }
    return dst;
}

__global__ void __launch_bounds__(64) k_near_src_fill(NearItem *items, const Range *__restrict__ ranges,
                                                      const int64_t *__restrict__ off, int32_t *near_src)
{
    const NearItem it = items[blockIdx.x];
    const int64_t o = off[blockIdx.x];
    if (threadIdx.x == 0) items[blockIdx.x].src_off = o;
    int32_t *dst = list_ranges(ranges, it.a_beg, it.a_end, near_src + o, [](int32_t c) { return !(c & FSS_SELF_BIT); });
    list_ranges(ranges, it.a_beg, it.a_end, dst, [](int32_t c) { return (c & FSS_SELF_BIT) != 0; });
}

// The near kernel hands each XCD a contiguous eighth of the items; inside every
// eighth, windows of NEAR_WINDOW items (about one round of the XCD's wave slots,
// whose sources fit its L2) go longest first, so the last wave slots to free
// hold short items.  Cost of an item: its sources over the phases of a 4-target
// tile.  One block ranks a window (equal costs keep their order).
constexpr int NEAR_WINDOW = 512;
__global__ void __launch_bounds__(NEAR_WINDOW) k_near_order(NearItem *items, int64_t n, int wpe)
{
    // cost, then place (earlier first): distinct keys, 0 beyond the window's end.
    // Whole unrolled rounds, so that their LDS reads are in flight together
    // (32 us with a read per turn of a loop of c turns).
    __shared__ __align__(16) uint64_t key[NEAR_WINDOW];
    const int64_t q8 = n >> 3, r8 = n & 7;
    const int64_t xcd = blockIdx.x / wpe, win = blockIdx.x % wpe;
    const int64_t b = xcd * q8 + min(xcd, r8) + win * NEAR_WINDOW, e = (xcd + 1) * q8 + min(xcd + 1, r8);
    const int c = (int)max((int64_t)0, min((int64_t)NEAR_WINDOW, e - b)), i = threadIdx.x;
    NearItem it{};
    uint64_t mine = 0;
    if (i < c) {
        it = items[b + i];
        const int tt = (it.tgt_cnt + 3) / 4, ph = 64 / tt;
        mine = (uint64_t)(((int64_t)it.n_other + it.n_self + ph - 1) / ph) * NEAR_WINDOW + (NEAR_WINDOW - 1 - i);
    }
    key[i] = mine;
    __syncthreads();
    int rank = 0;
#pragma unroll 16
    for (int j = 0; j < NEAR_WINDOW; j++) rank += key[j] > mine ? 1 : 0;
    if (i < c) items[b + rank] = it;
}

// Source list of every proxy item: the records of its class-B ranges in order.
// nitems: number of items where the host does not know it yet, or null.
__global__ void __launch_bounds__(64) k_far_src_count(const ProxyItem *__restrict__ items, const int *nitems,
                                                      const Range *__restrict__ ranges, int64_t *cnt)
{
    const int lane = threadIdx.x;
    int c = 0;
    if (!nitems || (int)blockIdx.x < *nitems) {
        const ProxyItem it = items[blockIdx.x];
        for (int r = it.b_beg + lane; r < it.b_end; r += 64) c += ranges[r].count & ~FSS_SELF_BIT;
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (lane == 0) cnt[blockIdx.x] = c;
}

__global__ void __launch_bounds__(64) k_far_src_fill(const ProxyItem *__restrict__ items, const int *nitems,
                                                     const Range *__restrict__ ranges,
                                                     const int64_t *__restrict__ off, int32_t *far_src)
{
    if (nitems && (int)blockIdx.x >= *nitems) return;
    const ProxyItem it = items[blockIdx.x];
    list_ranges(ranges, it.b_beg, it.b_end, far_src + off[blockIdx.x], [](int32_t) { return true; });
}

// Upward items: each charge node's records (main range, then exception range)
// in chunks of FSS_UP_CHUNK, in node order, the items of at most 32 records
// first (the upward pass runs them two per wave).  Per node: small items, others,
// whether it has several, and then their partial moments; an empty node has one
// empty item (zero charges).
__global__ void k_up_count(const int32_t *__restrict__ charge, int64_t nc, const int4 *__restrict__ nrange, int4 *per)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q > nc) return;
    int4 c = make_int4(0, 0, 0, 0);
    if (q < nc) {
        const int4 r = nrange[charge[q]];
        for (int part = 0; part < 2; part++) {
            const int32_t cnt = part ? r.w : r.y, tail = cnt % FSS_UP_CHUNK;
            const bool small = tail > 0 && tail <= 32;
            c.x += small ? 1 : 0;
            c.y += cnt / FSS_UP_CHUNK + (tail > 32 ? 1 : 0);
        }
        if (c.x + c.y == 0) c.x = 1;
        if (c.x + c.y > 1) {
            c.z = 1;
            c.w = c.x + c.y;
        }
    }
    per[q] = c;
}

__global__ void k_up_fill(const int32_t *__restrict__ charge, int64_t nc, const int4 *__restrict__ nrange,
                          const int4 *__restrict__ pos, int4 *items, int4 *multi)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nc) return;
    const int32_t g = charge[q];
    const int4 r = nrange[g], at = pos[q], nx = pos[q + 1];
    const bool several = nx.z > at.z;
    int32_t si = at.x, li = pos[nc].x + at.y, part = at.w;
    for (int h = 0; h < 2; h++) {
        const int32_t start = h ? r.z : r.x, cnt = h ? r.w : r.y;
        for (int32_t o = 0; o < cnt; o += FSS_UP_CHUNK) {
            const int32_t c = min(FSS_UP_CHUNK, cnt - o);
            items[c <= 32 ? si++ : li++] = make_int4(g, start + o, c, several ? part++ : -1);
        }
    }
    if (r.y + r.w == 0) items[si] = make_int4(g, 0, 0, -1);
    if (several) multi[at.z] = make_int4(g, at.w, nx.w, 0);
}

fss_status plan_finish(fss_ctx *ctx)
{
    Tree &T = ctx->tree;
    BuildScratch &B = ctx->build;
    hipStream_t s = ctx->stream;
    BuildInfo *info = B.info.as<BuildInfo>();
    if (T.batched) {
        FSS_TRY(T.tinv.ensure(sizeof(double) * 9 * std::max<int64_t>(1, T.nn)));
        hipLaunchKernelGGL(k_tinv, dim3((unsigned)div_up(T.nn, 256)), dim3(256), 0, s, T.tri_xyz.as<double>(), T.nn,
                           T.tinv.as<double>());
        T.d_xyz = T.tri_xyz.as<double>();
        T.d_info = T.tri_info.as<double>();
        T.d_tinv = T.tinv.as<double>();
    }
    // near-item source lists
    FSS_TRY(T.near_src.ensure(sizeof(int32_t) * std::max<int64_t>(1, T.n_near_src)));
    if (T.n_near > 0) {
        FSS_TRY(B.cnt.ensure(sizeof(int64_t) * T.n_near));
        FSS_TRY(B.off.ensure(sizeof(int64_t) * T.n_near));
        hipLaunchKernelGGL(k_near_src_count, dim3((unsigned)T.n_near), dim3(64), 0, s, T.near_items.as<NearItem>(),
                           T.ranges_a.as<Range>(), B.cnt.as<int64_t>());
        FSS_TRY(cub_exclusive_sum(B.cub, B.cnt.as<int64_t>(), B.off.as<int64_t>(), T.n_near, s));
        hipLaunchKernelGGL(k_near_src_fill, dim3((unsigned)T.n_near), dim3(64), 0, s, T.near_items.as<NearItem>(),
                           T.ranges_a.as<Range>(), B.off.as<int64_t>(), T.near_src.as<int32_t>());
        const int wpe = (int)div_up((T.n_near >> 3) + 1, NEAR_WINDOW);
        hipLaunchKernelGGL(k_near_order, dim3((unsigned)(8 * wpe)), dim3(NEAR_WINDOW), 0, s, T.near_items.as<NearItem>(),
                           T.n_near, wpe);
        FSS_HIP(hipGetLastError());
    }
    // proxy-item source lists; far_off[n_proxy] = total
    if (T.n_proxy > 0) {
        const int *nitems = T.batched ? nullptr : &info->n_proxy; // n_proxy is an upper bound until the end of a build
        FSS_TRY(B.cnt.ensure(sizeof(int64_t) * (T.n_proxy + 1)));
        FSS_TRY(T.far_off.ensure(sizeof(int64_t) * (T.n_proxy + 1)));
        FSS_TRY(T.far_src.ensure(sizeof(int32_t) * std::max<int64_t>(1, T.n_far_src)));
        FSS_HIP(hipMemsetAsync(B.cnt.as<int64_t>() + T.n_proxy, 0, sizeof(int64_t), s));
        hipLaunchKernelGGL(k_far_src_count, dim3((unsigned)T.n_proxy), dim3(64), 0, s, T.proxy_items.as<ProxyItem>(),
                           nitems, T.ranges_b.as<Range>(), B.cnt.as<int64_t>());
        FSS_TRY(cub_exclusive_sum(B.cub, B.cnt.as<int64_t>(), T.far_off.as<int64_t>(), T.n_proxy + 1, s));
        hipLaunchKernelGGL(k_far_src_fill, dim3((unsigned)T.n_proxy), dim3(64), 0, s, T.proxy_items.as<ProxyItem>(),
                           nitems, T.ranges_b.as<Range>(), T.far_off.as<int64_t>(), T.far_src.as<int32_t>());
        FSS_HIP(hipGetLastError());
    }
    // upward items: at most two short tails per charge node and one item per
    // FSS_UP_CHUNK records of a level
    T.n_up = T.n_up_multi = T.n_up_partial = T.n_up_small = 0;
    if (T.n_charge > 0) {
        const int64_t room = 2 * T.n_charge + (int64_t)T.L * (T.p0 / FSS_UP_CHUNK + 1);
        FSS_TRY(B.per.ensure(sizeof(int4) * (T.n_charge + 1)));
        FSS_TRY(B.pos.ensure(sizeof(int4) * (T.n_charge + 1)));
        FSS_TRY(T.up_items.ensure(sizeof(int4) * room));
        FSS_TRY(T.up_multi.ensure(sizeof(int4) * T.n_charge));
        hipLaunchKernelGGL(k_up_count, dim3((unsigned)div_up(T.n_charge + 1, 256)), dim3(256), 0, s,
                           T.charge_nodes.as<int32_t>(), T.n_charge, T.nrange.as<int4>(), B.per.as<int4>());
        FSS_TRY(cub_exclusive_add4(B.cub, B.per.as<int4>(), B.pos.as<int4>(), T.n_charge + 1, s));
        hipLaunchKernelGGL(k_up_fill, dim3((unsigned)div_up(T.n_charge, 256)), dim3(256), 0, s,
                           T.charge_nodes.as<int32_t>(), T.n_charge, T.nrange.as<int4>(), B.pos.as<int4>(),
                           T.up_items.as<int4>(), T.up_multi.as<int4>());
        FSS_HIP(hipMemcpyAsync(&info->up, B.pos.as<int4>() + T.n_charge, sizeof(int4), hipMemcpyDeviceToDevice, s));
        FSS_HIP(hipGetLastError());
    }
    FSS_TRY(proxy_records(ctx));
    BuildInfo h;
    FSS_TRY(read_back(ctx, &h, info, sizeof(h)));
    if (!T.batched) T.n_proxy = T.n_slot > 0 ? h.n_proxy : 0;
    if (T.n_charge > 0) {
        T.n_up_small = h.up.x;
        T.n_up = (int64_t)h.up.x + h.up.y;
        T.n_up_multi = h.up.z;
        T.n_up_partial = h.up.w;
    }
    return FSS_OK;
}

// the reference's node lists, needed by nothing else: particles of every level
// sorted by node (stable: ascending ids), the nodes' starts from their lengths
static fss_status export_lists(fss_ctx *ctx, int32_t *offsets, int32_t *ids)
{
    Tree &T = ctx->tree;
    hipStream_t s = ctx->stream;
    const int64_t n = T.n;
    DevBuf off, keys, sorted, vals, out, tmp;
    FSS_TRY(off.ensure(sizeof(int32_t) * T.nn));
    FSS_TRY(cub_exclusive_sum(tmp, T.counts.as<int32_t>(), off.as<int32_t>(), T.nn, s));
    if (offsets) FSS_TRY(read_back(ctx, offsets, off.p, sizeof(int32_t) * T.nn));
    if (!ids) return FSS_OK;
    FSS_TRY(keys.ensure(sizeof(uint32_t) * n));
    FSS_TRY(sorted.ensure(sizeof(uint32_t) * n));
    FSS_TRY(vals.ensure(sizeof(int32_t) * n));
    FSS_TRY(out.ensure(sizeof(int32_t) * n));
    int64_t base = 0;
    for (int l = 0; l < T.L; l++) {
        const int64_t cnt = n - T.stats.dropped[l];
        hipLaunchKernelGGL(k_level_keys, dim3((unsigned)div_up(n, 256)), dim3(256), 0, s,
                           T.loc.as<int32_t>() + (int64_t)l * n, T.found.as<uint8_t>() + (int64_t)l * n, n,
                           (uint32_t)level_size(l), keys.as<uint32_t>(), vals.as<int32_t>());
        FSS_TRY(cub_sort_pairs(tmp, keys.as<uint32_t>(), sorted.as<uint32_t>(), vals.as<int32_t>(), out.as<int32_t>(),
                               n, bits_for64((uint64_t)level_size(l)), s));
        if (cnt > 0) FSS_TRY(read_back(ctx, ids + base, out.p, sizeof(int32_t) * cnt));
        base += cnt;
    }
    return FSS_OK;
}

fss_status tree_export(fss_ctx *ctx, int32_t *loc, uint8_t *found, int32_t *counts, int32_t *offsets,
                       int32_t *ids, int32_t *inter, double *tri_info, double *tri_xyz)
{
    Tree &T = ctx->tree;
    if (!T.built) {
        set_error("tree_export before tree_build");
        return FSS_ERR_STATE;
    }
    if (T.batched) {
        set_error("tree_export is not available for a batch");
        return FSS_ERR_STATE;
    }
    if (loc) FSS_TRY(read_back(ctx, loc, T.loc.p, sizeof(int32_t) * T.L * T.n));
    if (found) FSS_TRY(read_back(ctx, found, T.found.p, (size_t)T.L * T.n));
    if (counts) FSS_TRY(read_back(ctx, counts, T.counts.p, sizeof(int32_t) * T.nn));
    if (offsets || (ids && T.nlist > 0)) FSS_TRY(export_lists(ctx, offsets, T.nlist > 0 ? ids : nullptr));
    if (inter && T.ninter > 0) FSS_TRY(read_back(ctx, inter, T.inter.p, sizeof(int32_t) * 7 * T.ninter));
    if (tri_info) FSS_TRY(read_back(ctx, tri_info, T.d_info, sizeof(double) * 4 * T.ntri_all));
    if (tri_xyz) FSS_TRY(read_back(ctx, tri_xyz, T.d_xyz, sizeof(double) * 9 * T.ntri_all));
    return FSS_OK;
}

} // namespace fss
