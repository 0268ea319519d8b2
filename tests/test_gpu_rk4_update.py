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
