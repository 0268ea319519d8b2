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


def _slabs(n):
    """Rows of every slab of the sum over n particles and how its units are cut
    (one unit a run, equal runs, or long and short ones): sym_slab's arithmetic, with
    the workspace that the source gives it."""
    import os
    import re
    from conftest import ROOT
    src = open(os.path.join(ROOT, "fast-sphere-sum_amd", "csrc", "fss_direct.hip")).read()
    room = (int(re.search(r"SYM_BYTES = \(int64_t\)(\d+) << 20", src).group(1)) << 20) // 24
    R = 2 if n < 18000 else 4
    T, RT, slots, K = 256 * R, 4 * R, 768 if R == 4 else 1024, -(-n // 64)
    rows, r0, out = -(-n // T), 0, []

    def cols(r):
        return (r - r0) * 64 * K - T * (r * (r + 1) - r0 * (r0 + 1)) // 2

    while r0 < rows:
        r1 = r0 + 1
        while r1 < rows and cols(r1 + 1) + (r1 + 1 - r0 + slots) * T <= room:
            r1 += 1
        units = (r1 - r0) * K - RT * (r1 * (r1 - 1) - r0 * (r0 - 1)) // 2
        runs = (room - cols(min(r1, rows - 1))) // T - (r1 - r0)
        out.append((r1 - r0, "one" if units <= min(2 * slots, runs) else "equal" if runs < 2 * slots else "long"))
        r0 = r1
    return out


# particles, and the slabs that they are meant to take (asserted below, so that
# another workspace does not leave a cut untested)
SLABS = {50021: ["equal"], 62208: ["equal"], 62209: ["equal", "one"], 70001: ["equal", "long"],
         100003: ["equal"] * 3}


def _sampled(orc, c, m=400):
    idx = np.unique(np.concatenate([np.random.default_rng(1).integers(0, len(c[0]), m), [0, len(c[0]) - 1]]))
    return idx, orc.rhs_direct(*c, idx=idx, nthreads=8)


@pytest.mark.parametrize("n", sorted(SLABS))
def test_pair_sum_in_slabs_matches_oracle(fsslib, orc, n):
    """One and several slabs of rows, and each cut of a slab's units; the
    allocation-free entry takes the same plan, so the same bits."""
    assert [k for _, k in _slabs(n)] == SLABS[n]
    c = _case(n, 6)
    print(f"direct pairs n={n} slabs={_slabs(n)}", flush=True)
    d = _dev(*c)
    ctx = fsslib.Context()
    got = [t.cpu().numpy() for t in ctx.velocity_direct(*d)]
    idx, ref = _sampled(orc, c)
    assert _err([g[idx] for g in got], ref) <= 1e-12
    for g, h in zip(got, ctx.velocity_direct_noalloc(*d)):
        np.testing.assert_array_equal(g, h.cpu().numpy())


@pytest.mark.parametrize("shift", [0, 37])
def test_pair_sum_outputs_over_inputs_in_slabs(fsslib, orc, shift):
    """Outputs over the inputs, element by element and shifted: with several slabs
    the inputs are read again after the first velocities are known."""
    n = 70001
    assert len(_slabs(n)) > 1
    c = _case(n, 6)
    buf = [t.new_zeros(n + shift) for t in _dev(*c[:4])]
    d = [b[:n] for b in buf]
    for a, b in zip(d, _dev(*c[:4])):
        a.copy_(b)
    out = [buf[k][shift:] for k in (3, 0, 1, 2)]
    got = [t.cpu().numpy() for t in fsslib.Context().velocity_direct(*d, *_dev(c[4]), out=out)]
    idx, ref = _sampled(orc, c)
    assert _err([g[idx] for g in got], ref) <= 1e-12


@pytest.mark.parametrize("n", [5003, 20011, 70001])
@pytest.mark.parametrize("first", ["apart", "over"])
def test_captured_call_with_other_outputs(fsslib, n, first):
    """An eager call sizes the workspace for a captured one of as many particles,
    whether the outputs of either overlap the inputs (another kernel) or not."""
    import torch
    s = torch.cuda.Stream()
    d = _dev(*_case(n, 6))
    ctx = fsslib.Context(stream=s)
    spare = [t.clone() for t in d[:4]]
    want = [t.clone() for t in fsslib.Context().velocity_direct(*d)]
    into = [torch.empty_like(t) for t in spare]
    torch.cuda.synchronize()
    print(f"direct pairs captured n={n} first={first}", flush=True)

    def call(over):
        # the inputs of a call over them are set again before each
        x = spare if over else d[:4]
        return ctx.velocity_direct(*x, d[4], out=spare if over else into)

    call(first == "over")
    torch.cuda.synchronize()
    for a, b in zip(spare, d):
        a.copy_(b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        got = call(first != "over")
    for _ in range(3):
        for a, b in zip(spare, d):
            a.copy_(b)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert _err([t.cpu().numpy() for t in got], [t.cpu().numpy() for t in want]) <= 1e-12


@pytest.mark.parametrize("precision,eager,captured", [
    (0, (20011, None), (15001, None)), (0, (60000, None), (45001, None)), (0, (2700, None), (2561, None)),
    (0, (3350, None), (3250, None)), (1, (655361, None), (300001, None)), (1, (40000, None), (30011, None)),
    (0, (20011, 100), (20011, 7001)), (0, (20011, 20011), (20011, 3001)), (0, (900001, None), (900001, 20011))])
def test_captured_call_of_fewer_particles(fsslib, precision, eager, captured):
    """An eager call sizes the workspace for every later one of as many particles or
    fewer, whatever its targets: layouts differ, and a smaller sum may cut itself
    into more runs."""
    import torch
    s = torch.cuda.Stream()
    ctx = fsslib.Context(stream=s, precision=precision)
    rng = np.random.default_rng(3)
    print(f"direct captured precision={precision} eager={eager} captured={captured}", flush=True)

    def case(n, m):
        d = _dev(*_case(n, 6))
        if m is None:
            return lambda c: c.velocity_direct(*d)
        idx = torch.from_numpy(rng.integers(0, n, m)).cuda()
        return lambda c: c.velocity_direct_targets(*d, idx)

    big, small = case(*eager), case(*captured)
    want = [t.cpu().numpy() for t in small(fsslib.Context(precision=precision))]
    torch.cuda.synchronize()
    big(ctx)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        got = small(ctx)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g.cpu().numpy(), w)
