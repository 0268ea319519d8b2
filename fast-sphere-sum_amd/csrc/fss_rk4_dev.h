// fss_rk4_dev.h -- the RK4 update of one particle, taken by the last kernel of a
// velocity evaluation with the velocities in registers.  As kernels of their own
// the updates read them, the state and (at the end) all four stages again: 46 us a
// stage and 107 a step of 3.05 M particles, and 5 us each for 10,242, of 24 between
// a step's kernels.
#pragma once

#include "fss_internal.h"

namespace fss {

// proj = project_points (Old-BVE-code/helpers.h:362-372): x <- x/|x| and
// omega += -2 Omega (z_new - z_old), which keeps omega + 2 Omega z per particle.
// No FMA contraction: every product and sum of the update is rounded separately,
// as the reference's scalar_mult and vec_add round them.
__device__ inline void project_one(double &x, double &y, double &z, double &vort, double omega)
{
#pragma clang fp contract(off)
    // project_to_sphere(p, 1.0): p[i] *= 1.0 / norm (helpers.h:82-85)
    double s = 0.0;
    s += x * x;
    s += y * y;
    s += z * z;
    double nrm = sqrt(s);
    double f = 1.0 / nrm;
    double px = x * f, py = y * f, pz = z * f;
    double dz = pz - z;
    x = px;
    y = py;
    z = pz;
    vort += -2 * omega * dz;
}

// Particle i with the velocities k of this stage: the next stage's state
// ys = proj(y + fac k) (new_dynamics.cpp:174-184), or at the end of the step
// y = proj(y + fac (k1 + 2 k2 + 2 k3 + k4)), fac = dt / 6 (new_dynamics.cpp:205-229)
__device__ inline void rk_next(const RkNext &r, int64_t i, double k0, double k1, double k2, double k3)
{
#pragma clang fp contract(off)
    if (r.mode == RkNext::NONE) return;
    double v[4] = {k0, k1, k2, k3};
    double *f[4] = {r.x, r.y, r.z, r.vort};
    if (r.mode == RkNext::STAGE) {
        for (int c = 0; c < 4; c++) v[c] = v[c] * r.fac + f[c][i];
    } else {
        for (int c = 0; c < 4; c++) {
            double a = r.k[c * r.n + i];
            a += r.k[4 * r.n + c * r.n + i] * 2;
            a += r.k[8 * r.n + c * r.n + i] * 2;
            a += v[c];
            a *= r.fac;
            v[c] = f[c][i] + a;
        }
    }
    project_one(v[0], v[1], v[2], v[3], r.omega);
    for (int c = 0; c < 4; c++) (r.mode == RkNext::STAGE ? r.ys + c * r.n : f[c])[i] = v[c];
}

} // namespace fss
