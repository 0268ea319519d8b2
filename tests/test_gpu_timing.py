"""GPU: the stage times that a context reads back, over calls on several streams."""
import ctypes

import pytest

from test_gpu_direct_layouts import _case, _dev

pytestmark = pytest.mark.gpu


def test_mean_waits_for_every_stream_of_the_window(fsslib):
    """A long call on one stream, a short one on another: the means read at once are
    those read after both have ended.  (The tree's workspace is apart from the direct
    sum's, so the two calls may overlap.)"""
    import torch
    big, small = _dev(*_case(200003)), _dev(*_case(2001))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    ctx = fsslib.Context(stream=a, tree_levels=3, eval_mode=1, assign_mode=1, node_rule=1)
    ctx.tree_build(*small[:3])
    ctx.velocity_direct(*big)
    ctx.velocity_tree(*small)
    torch.cuda.synchronize()
    ctx.timing_reset()
    ctx.velocity_direct(*big)
    fsslib._check(fsslib.lib().fss_set_stream(ctx.h, ctypes.c_void_p(b.cuda_stream)))
    ctx.velocity_tree(*small)
    at_once = ctx.timing_mean(), ctx.timing_far_mean()
    torch.cuda.synchronize()
    print("mean ms read at once", at_once, "after", ctx.timing_mean(), flush=True)
    assert at_once == (ctx.timing_mean(), ctx.timing_far_mean())
