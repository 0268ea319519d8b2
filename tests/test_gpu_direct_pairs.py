"""GPU: the FP64 direct sum over unordered pairs (rows of 512 or 1,024 targets,
tiles of 64 sources, slabs of rows) against the oracle's direct sum, at sizes
around its first size, its change of layout, the row, tile and slab edges.

Points are a Fibonacci lattice, so the bar of the other direct-sum tests
applies: rel-L2 <= 1e-12 (the device and the oracle round 1 - x.y alike; the rest
is the reciprocals' last bits and summation order)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_direct_layouts import _case, _dev, _err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3299, 3300, 3584, 3585, 3648, 17999, 18000, 18432, 18433, 41023])
def test_pair_sum_matches_oracle(fsslib, orc, n):
    c = _case(n, 6)
    print(f"direct pairs n={n}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct(*_dev(*c))]
    assert _err(got, orc.rhs_direct(*c, nthreads=8)) <= 1e-12


@pytest.mark.parametrize("n", [5003, 20011])
def test_pair_sum_coincident_points(fsslib, orc, n):
    """Coincident points of different rows (1 - x.y exactly zero) get no finite
    velocity, as in the reference; every other particle is as the oracle has it."""
    c = [a.copy() for a in _case(n, 4)]
    i, j = 5, n - 100
    for a, v in zip(c[:3], (0.0, 0.6, 0.8)):
        a[i] = a[j] = v
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct(*_dev(*c))]
    ref = orc.rhs_direct(*c, nthreads=8)
    keep = np.ones(n, bool)
    keep[[i, j]] = False
    assert _err([g[keep] for g in got], [r[keep] for r in ref]) <= 1e-12
    for g, r in zip(got[:3], ref[:3]):
        assert np.isfinite(g[[i, j]]).tolist() == np.isfinite(r[[i, j]]).tolist()


def test_pair_sum_outputs_over_inputs(fsslib, orc):
    """Outputs that share the inputs' memory are written last, as before."""
    n = 41023
    c = _case(n, 6)
    d = _dev(*c)
    got = fsslib.Context().velocity_direct(*d, out=(d[3], d[0], d[1], d[2]))
    assert _err([t.cpu().numpy() for t in got], orc.rhs_direct(*c, nthreads=8)) <= 1e-12


@pytest.mark.parametrize("n", [41023, 70001])
def test_pair_sum_outputs_over_each_other(fsslib, orc, n):
    """One array for two outputs (a caller without use for one of them) holds the
    component written last, and the others are as with arrays of their own."""
    c = _case(n, 6)
    d = _dev(*c)
    ctx = fsslib.Context()
    want = [t.clone() for t in ctx.velocity_direct(*d)]
    for pick in ((0, 1, 2, 2), (0, 0, 2, 3), (0, 1, 1, 3), (0, 1, 2, 0)):
        buf = [want[0].new_full((n,), float("nan")) for _ in range(4)]
        got = ctx.velocity_direct(*d, out=[buf[k] for k in pick])
        for k in range(4):
            last = max(j for j in range(4) if pick[j] == pick[k])
            assert rel_l2(got[k].cpu().numpy(), want[last].cpu().numpy()) <= 1e-12, (pick, k)
