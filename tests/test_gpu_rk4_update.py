"""GPU: the RK4 update that the last kernel of a direct sum takes, in every layout
of the sum (pairs in one and several slabs, runs, whole groups), against the step
put together from velocity calls.

Both round the same products and sums of numbers of order one to ten, four stages
of about ten operations each at 1.1e-16: 1e-14 absolute."""
import numpy as np
import pytest

from test_gpu_direct_layouts import _case, _dev

pytestmark = pytest.mark.gpu
OMEGA = 2 * np.pi


def _project(y):
    r = 1.0 / (y[0] * y[0] + y[1] * y[1] + y[2] * y[2]).sqrt()
    p = [c * r for c in y[:3]]
    return p + [y[3] - 2 * OMEGA * (p[2] - y[2])]


@pytest.mark.parametrize("n,precision", [(700, 0), (5003, 0), (41023, 0), (20011, 1), (655362, 1)])
def test_direct_step_equals_its_stages(fsslib, n, precision):
    d = _dev(*_case(n, 8))
    dt = 0.01
    ctx = fsslib.Context(precision=precision)
    print(f"rk4 update n={n} precision={precision}", flush=True)
    y, area, k = d[:4], d[4], []
    s = y
    for f in (dt / 2, dt / 2, dt, None):
        k.append([t.clone() for t in ctx.velocity_direct(*[c.contiguous() for c in s], area)])
        if f is not None:
            s = _project([kc * f + c for kc, c in zip(k[-1], y)])
    want = _project([c + (a + b * 2 + e * 2 + g) * (dt / 6) for c, a, b, e, g in zip(y, *k)])
    got = [t.clone() for t in y]
    ctx.rk4_step(*got, area, dt)
    for g, w in zip(got, want):
        assert float((g - w).abs().max()) <= 1e-14


@pytest.mark.parametrize("n", [62209, 100003])
def test_direct_step_in_slabs_equals_its_stages(fsslib, n):
    """The update of a target is taken with its own row's slab, while later slabs
    still read the others' state."""
    from test_gpu_direct_pairs import _slabs
    assert len(_slabs(n)) > 1
    test_direct_step_equals_its_stages(fsslib, n, 0)


@pytest.mark.parametrize("evalm,precision", [(0, 0), (1, 0), (1, 1)])
def test_tree_step_with_exception_records_equals_its_stages(fsslib, evalm, precision):
    """Particles on lists outside their main path have records of their own, and the
    step then runs in the caller's order; the graph's replays are the same step."""
    x, y, z, tris = fsslib.grid_icosahedral(5)
    d = _dev(x, y, z, fsslib.rossby_haurwitz(x, y, z)[0], fsslib.third_areas(x, y, z, tris))
    dt = 0.01
    ctx = fsslib.Context(precision=precision, tree_levels=6, eval_mode=evalm, assign_mode=0, node_rule=evalm)
    ctx.tree_build(*d[:3])
    assert ctx.stats().n_records > len(x)
    print(f"rk4 tree exceptions mode={evalm} precision={precision} records={ctx.stats().n_records}", flush=True)
    y0, area, k = d[:4], d[4], []
    s = y0
    for f in (dt / 2, dt / 2, dt, None):
        k.append([t.clone() for t in ctx.velocity_tree(*[c.contiguous() for c in s], area)])
        if f is not None:
            s = _project([kc * f + c for kc, c in zip(k[-1], y0)])
    want = _project([c + (a + b * 2 + e * 2 + g) * (dt / 6) for c, a, b, e, g in zip(y0, *k)])
    got = [t.clone() for t in y0]
    ctx.rk4_step(*got, area, dt, use_tree=True)
    # in mixed precision an ulp of a stage's state is one FP32 ulp of an offset here and there
    for g, w in zip(got, want):
        assert float((g - w).abs().max()) <= (1e-14 if precision == 0 else 1e-9)
    ref, run = [t.clone() for t in y0], [t.clone() for t in y0]
    for _ in range(3):
        ctx.rk4_step(*ref, area, dt, use_tree=True)
    ctx.rk4_run_graph(*run, area, dt, 3, use_tree=True)
    for g, w in zip(run, ref):
        np.testing.assert_array_equal(g.cpu().numpy(), w.cpu().numpy())
