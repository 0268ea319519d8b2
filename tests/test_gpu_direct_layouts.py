"""GPU: the direct sum's work layouts (one, two or four targets per lane,
tiles of 16, 64 or 256 sources, cut into runs over the blocks or a whole target
group per block) against the oracle's direct sum, at sizes around the tile,
wave and group edges and where the layout changes.

Points are a Fibonacci lattice (separated by about 3.5/sqrt(n)), so the bars of
the other direct-sum tests apply: FP64 rel-L2 <= 1e-12 (the device and the
oracle round 1 - x.y alike; the rest is summation order), mixed <= 1e-6."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _case(n, seed=1):
    k = np.arange(n) + 0.5
    z = 1 - 2 * k / n
    t = np.pi * (1 + 5 ** 0.5) * k
    r = np.sqrt(1 - z * z)
    x, y = r * np.cos(t), r * np.sin(t)
    q = 1 / np.sqrt(x * x + y * y + z * z)
    rng = np.random.default_rng(seed)
    return x * q, y * q, z * q, rng.normal(size=n), np.full(n, 4 * np.pi / n)


def _dev(*arrs):
    import torch
    return [torch.from_numpy(np.ascontiguousarray(a)).to("cuda") for a in arrs]


def _err(got, ref):
    return max(rel_l2(np.stack(got[:3], 1), np.stack(ref[:3], 1)), rel_l2(got[3], ref[3]))


@pytest.mark.parametrize("precision,bar", [(0, 1e-12), (1, 1e-6)])
@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 65, 255, 256, 257, 1025, 2561, 7001, 9000, 16385, 20011])
def test_direct_layouts_match_oracle(fsslib, orc, n, precision, bar):
    c = _case(n)
    print(f"direct n={n} precision={precision}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context(precision=precision).velocity_direct(*_dev(*c))]
    ref = orc.rhs_direct(*c, nthreads=8)
    assert _err(got, ref) <= bar


@pytest.mark.parametrize("n,m", [(300, 1), (5000, 65), (20011, 300), (20011, 2000), (40, 655361)])
def test_direct_targets_layouts_match_oracle(fsslib, orc, n, m):
    """Targets in any order, repeated (m > n) and, at m = 655,361, in whole
    target groups per block: each equals its row of the full sum."""
    import torch
    c = _case(n, 2)
    idx = np.random.default_rng(3).integers(0, n, m)
    print(f"direct targets n={n} m={m}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct_targets(*_dev(*c), torch.from_numpy(idx))]
    ref = [r[idx] for r in orc.rhs_direct(*c, nthreads=8)]
    assert _err(got, ref) <= 1e-12


@pytest.mark.parametrize("n", [200, 20011])
def test_direct_coincident_points(fsslib, orc, n):
    """A pair of coincident points whose 1 - x.y is exactly zero (the reference
    divides by it: the two get no finite velocity) leaves every other target,
    those of the same lane included, as the oracle has it."""
    c = [a.copy() for a in _case(n, 4)]
    i, j = 5, 5 + 64 * 3
    for a, v in zip(c[:3], (0.0, 0.6, 0.8)):
        a[i] = a[j] = v
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct(*_dev(*c))]
    ref = orc.rhs_direct(*c, nthreads=8)
    keep = np.ones(n, bool)
    keep[[i, j]] = False
    assert _err([g[keep] for g in got], [r[keep] for r in ref]) <= 1e-12
    for g, r in zip(got[:3], ref[:3]):
        assert np.isfinite(g[[i, j]]).tolist() == np.isfinite(r[[i, j]]).tolist()


@pytest.mark.parametrize("n,precision,bar", [(33, 0, 1e-12), (47, 0, 1e-12), (300, 1, 1e-6), (513, 1, 1e-6), (767, 1, 1e-6)])
def test_direct_groups_of_few_tiles_match_oracle(fsslib, orc, n, precision, bar):
    """Two or three tiles a target group: a block per group."""
    c = _case(n, 5)
    print(f"direct few tiles n={n} precision={precision}", flush=True)
    ctx = fsslib.Context(precision=precision)
    ref = orc.rhs_direct(*c, nthreads=8)
    for call in (ctx.velocity_direct, ctx.velocity_direct_noalloc):
        assert _err([t.cpu().numpy() for t in call(*_dev(*c))], ref) <= bar


@pytest.mark.parametrize("n,m", [(40, 40003), (40, 140001), (200, 400001)])
def test_direct_many_targets_of_few_tiles_match_oracle(fsslib, orc, n, m):
    """Few sources and more target groups than blocks: long and short runs over
    groups of three or four tiles."""
    import torch
    c = _case(n, 2)
    idx = np.random.default_rng(7).integers(0, n, m)
    print(f"direct targets few tiles n={n} m={m}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct_targets(*_dev(*c), torch.from_numpy(idx))]
    assert _err(got, [r[idx] for r in orc.rhs_direct(*c, nthreads=8)]) <= 1e-12


def _layout(n, m):
    """(targets a lane, sources a wave tile) of a call with chosen targets below
    655,361: direct_plan's choice from the measured table in the source."""
    import os
    import re
    from conftest import ROOT
    src = open(os.path.join(ROOT, "fast-sphere-sum_amd", "csrc", "fss_direct.hip")).read()
    table = re.search(r"kDirect64\[4\] = \{(.*?)\};", src, flags=re.S).group(1)
    lays = [[float(v) for v in r.split(",")] for r in re.findall(r"\{([^{}]*)\}", table)]
    R, wt, _, _ = min(lays, key=lambda a: a[2] + -(-m // (64 * a[0])) * 64 * a[0] * n / a[3])
    return int(R), int(wt)


@pytest.mark.parametrize("n,m,layout", [(20011, 301, (1, 16)), (20011, 1501, (1, 64)), (20011, 3001, (2, 64)),
                                        (60000, 6001, (4, 64)), (30011, 20011, (4, 64))])
def test_direct_targets_every_layout_matches_oracle(fsslib, orc, n, m, layout):
    import torch
    assert _layout(n, m) == layout
    c = _case(n, 2)
    idx = np.random.default_rng(8).permutation(n)[:m]
    print(f"direct targets n={n} m={m} layout={layout}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct_targets(*_dev(*c), torch.from_numpy(idx))]
    assert _err(got, orc.rhs_direct(*c, idx=idx, nthreads=8)) <= 1e-12


def test_direct_whole_groups_of_many_tiles(fsslib, orc):
    """A block per target group, which walks the tiles of 700 sources: 655,361
    targets in FP64."""
    import torch
    n = 700
    c = _case(n, 9)
    idx = np.random.default_rng(9).integers(0, n, 655361)
    print(f"direct whole groups n={n}", flush=True)
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct_targets(*_dev(*c), torch.from_numpy(idx))]
    assert _err(got, [r[idx] for r in orc.rhs_direct(*c, nthreads=8)]) <= 1e-12
