"""The tensors that the velocity calls return when the caller gives none."""
import torch


def _outputs(fsslib, m):
    ctx = fsslib.Context.__new__(fsslib.Context)  # no device needed to allocate on the host
    ctx.device = torch.device("cpu")
    return ctx._out(m)[0]


def test_outputs_are_tensors_of_their_own(fsslib):
    """Each component can be kept, saved, resized and changed by itself."""
    o = _outputs(fsslib, 5)
    assert len({t.untyped_storage().data_ptr() for t in o}) == 4
    assert all(t.untyped_storage().nbytes() == 40 and not t._is_view() for t in o)


def test_outputs_in_autograd(fsslib):
    """In-place arithmetic with a tensor that needs gradients, and on one
    component while another is saved for the backward pass."""
    p = torch.ones(5, dtype=torch.float64, requires_grad=True)
    u, v, w, d = (t.fill_(k + 1.0) for k, t in enumerate(_outputs(fsslib, 5)))
    u.add_(p)
    loss = (p * v).sum() + u.sum()
    w.mul_(2.0)
    loss.backward()
    torch.testing.assert_close(p.grad, torch.full((5,), 3.0, dtype=torch.float64))
