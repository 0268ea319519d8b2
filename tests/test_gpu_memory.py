"""GPU: device memory that a context holds after a build."""
import pytest

from test_gpu_direct_layouts import _case, _dev

pytestmark = pytest.mark.gpu


def _held(fsslib, c, levels, **kw):
    """Memory that a build takes beyond a context that has built a small tree (its
    queue's own memory, for kernels with a stack, comes with the first)."""
    import torch
    d, s = _dev(*c), _dev(*_case(40))
    ctx = fsslib.Context(eval_mode=1, assign_mode=1, node_rule=1, tree_levels=2, **kw)
    ctx.tree_build(*s[:3])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    ctx.autotune_levels(*d, levels, levels, reps=1)  # one depth: its tree, and one warm stage
    return ctx, free - torch.cuda.mem_get_info()[0]


def test_lists_are_sized_by_the_pairs_there_can_be(fsslib):
    """100 particles on 6 levels lie in at most 600 nodes, so there are at most
    360,000 interactions whatever theta allows: 40 MB of list at four times as many,
    and 50 MB of frontier."""
    ctx, held = _held(fsslib, _case(100), 6, theta=0.05)
    print(f"held {held / 1e6:.0f} MB for {ctx.stats().n_interactions} interactions", flush=True)
    assert held <= 200e6


def test_inverse_matrices_for_nodes_only(fsslib):
    """Triangles go one level deeper than the nodes: 104 bytes each of those, and per
    node the inverse matrix, cap, proxies, records and ranges (308 bytes at degree 1)."""
    L = 10
    ctx, held = _held(fsslib, _case(1000), L, degree=1, theta=0.7)
    nodes, tris = [20 * (4 ** k - 1) // 3 for k in (L, L + 1)]
    print(f"held {held / 1e9:.2f} GB", flush=True)
    assert held <= 1.1 * (104 * tris + 308 * nodes)
