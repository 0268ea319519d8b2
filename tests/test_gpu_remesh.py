"""GPU: remesh (libfss fss_remesh, through the C ABI) against the oracle's
restatement of regrid_points2 / tri_interp: the same containing triangle for
every grid point and the same interpolated vorticity and tracer."""
import numpy as np
import pytest

import oracle
from test_remesh_oracle import _advect

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,amp,drop", [(4, 0.01, 0), (5, 0.006, 0), (4, 0.02, 7)])
def test_remesh_matches_oracle(fsslib, level, amp, drop):
    import torch
    x, y, z, tris = fsslib.grid_icosahedral(level)
    off, idx = fsslib.vertex_triangles(len(x), tris)
    if drop:  # empty adjacency lists force the full search
        keep = np.ones(len(x), dtype=bool)
        keep[::drop] = False
        cnt = np.where(keep, np.diff(off), 0)
        idx = np.concatenate([idx[off[i]:off[i + 1]] for i in range(len(x)) if keep[i]]).astype(np.int32)
        off = np.zeros_like(off)
        off[1:] = np.cumsum(cnt)
    ax, ay, az = _advect(x, y, z, amp, seed=level)
    av = np.sin(3 * ax) * np.cos(2 * az) + 0.3 * ay
    tr = 2 + np.arcsin(az)
    want_v, want_t, want_tri, want_nf = oracle.remesh(ax, ay, az, av, tris, off, idx, x, y, z, atracer=tr)
    print(f"remesh level={level} amp={amp} drop={drop} n={len(x)} fallbacks={want_nf}", flush=True)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ctx = fsslib.Context()
    got_v, got_t, got_tri, nf = ctx.remesh(d(ax), d(ay), d(az), d(av), d(tris.astype(np.int32)), d(off), d(idx),
                                           d(x), d(y), d(z), atracer=d(tr), tri_out=True)
    assert nf == want_nf
    np.testing.assert_array_equal(got_tri.cpu().numpy(), want_tri)
    np.testing.assert_allclose(got_v.cpu().numpy(), want_v, rtol=0, atol=1e-15)
    np.testing.assert_allclose(got_t.cpu().numpy(), want_t, rtol=0, atol=1e-15)


def test_remesh_after_rk4_steps_conserves_circulation_roughly(fsslib):
    """Remesh of an advected Rossby-Haurwitz state: the grid vorticity stays
    close to the advected one (linear interpolation error) and the mean
    absolute vorticity is kept to the interpolation error."""
    import torch
    x, y, z, tris = fsslib.grid_icosahedral(4)
    area = fsslib.voronoi_areas(x, y, z, tris)
    v, _ = fsslib.rossby_haurwitz(x, y, z, 0.5, 0.5)
    off, idx = fsslib.vertex_triangles(len(x), tris)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    st = [d(a) for a in (x, y, z, v, area)]
    ctx = fsslib.Context()
    for _ in range(3):
        ctx.rk4_step(*st, 0.01)
    print("remesh after 3 RK4 steps, level 4", flush=True)
    vo, _, _, nf = ctx.remesh(st[0], st[1], st[2], st[3], d(tris.astype(np.int32)), d(off), d(idx), d(x), d(y),
                              d(z))
    vo = vo.cpu().numpy()
    adv = st[3].cpu().numpy()
    assert np.abs(vo - v).max() < 0.5 * np.abs(v).max()
    om = 2 * np.pi
    m0 = np.sum((adv + 2 * om * st[2].cpu().numpy()) * area)
    m1 = np.sum((vo + 2 * om * z) * area)
    assert abs(m1 - m0) < 1e-2 * np.sum(np.abs(adv) * area)


def _distorted(fsslib, kind):
    """Advected meshes whose triangles leave the bins of the full search: folded
    over (large displacement), collapsed and nearly collapsed edges (singular and
    ill-conditioned triangles), one patch shrunk so that its neighbours are
    stretched over many cells."""
    x, y, z, tris = fsslib.grid_icosahedral(4)
    p = np.stack((x, y, z), 1)
    rng = np.random.default_rng(11)
    p = p + 0.004 * rng.normal(size=p.shape)  # targets off the mesh edges
    if kind == "fold":
        p = p + 0.12 * rng.normal(size=p.shape)
    elif kind == "collapse":
        for k, t in enumerate(rng.choice(len(tris), 60, replace=False)):
            a, b, _ = tris[t]
            p[a] = p[b] + (0, 1e-14, 1e-9)[k % 3] * rng.normal(size=3)
    else:
        near = p @ p[0] > 0.9
        p[near] = p[0] + 0.02 * (p[near] - p[0])
    return (x, y, z), p / np.linalg.norm(p, axis=1)[:, None], tris


@pytest.mark.parametrize("kind", ["fold", "collapse", "stretch"])
def test_remesh_full_search_of_distorted_meshes(fsslib, kind):
    """No adjacency at all, so every target takes the full search: the same
    (lowest-index) triangle as the oracle's scan."""
    import torch
    (x, y, z), p, tris = _distorted(fsslib, kind)
    n = len(x)
    off, idx = np.zeros(n + 1, np.int32), np.zeros(1, np.int32)
    ax, ay, az = (np.ascontiguousarray(c) for c in p.T)
    av = np.sin(3 * ax) + 0.3 * ay
    want_v, _, want_tri, want_nf = oracle.remesh(ax, ay, az, av, tris, off, idx, x, y, z)
    print(f"remesh {kind}: n={n} fallbacks={want_nf}", flush=True)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got_v, _, got_tri, nf = fsslib.Context().remesh(d(ax), d(ay), d(az), d(av), d(tris.astype(np.int32)), d(off),
                                                    d(idx), d(x), d(y), d(z), tri_out=True)
    assert nf == want_nf == n
    np.testing.assert_array_equal(got_tri.cpu().numpy(), want_tri)
    np.testing.assert_allclose(got_v.cpu().numpy(), want_v, rtol=0, atol=1e-15 * np.abs(want_v).max())
