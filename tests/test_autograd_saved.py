"""Saved-tensor hooks and the site energies (CPU, the oracle behind the interface
of the device evaluator): the parameters that the second backward reaches are
those that the forward saved, also where hooks keep copies and the tensor has
been written to since (without hooks that is refused)."""
import numpy as np
import pytest
import torch

from acehip.autograd import site_energies
from test_autograd_host import _case


def _setup():
    ev, c, off, R = _case("Invariant", 3, 4)
    theta = torch.tensor(0.5 * c, requires_grad=True)
    x = torch.tensor(R.T.copy(), requires_grad=True)
    w = torch.tensor(np.random.default_rng(3).normal(size=tuple(x.shape)))
    return ev, off, theta, x, w


def _mixed(E, x, w, theta):
    (gx,) = torch.autograd.grad(E.sum(), x, create_graph=True)
    return torch.autograd.grad(gx, theta, w)[0]


def test_written_to_since_under_hooks():
    ev, off, theta, x, w = _setup()
    want = _mixed(site_energies(ev, 2.0 * theta, off, x), x, w, theta)
    c = 2.0 * theta
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().clone(), lambda t: t):
        E = site_energies(ev, c, off, x)
    c.mul_(3.0)  # a step of the graph that the energies do not know of
    assert torch.allclose(_mixed(E, x, w, theta), want, rtol=1e-13)
    c = 2.0 * theta
    E = site_energies(ev, c, off, x)
    c.mul_(3.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        _mixed(E, x, w, theta)


def test_parameters_without_gradient():
    ev, off, theta, x, w = _setup()
    c = (2.0 * theta).detach()
    E = site_energies(ev, c, off, x)
    (g,) = torch.autograd.grad(E.sum(), x, create_graph=True)
    (want,) = torch.autograd.grad(site_energies(ev, 2.0 * theta, off, x).sum(), x)
    assert torch.equal(g.detach(), want)


def test_positions_after_parameters_and_the_other_way():
    """Each gradient twice over, in either order, from one retained graph."""
    ev, off, theta, x, w = _setup()
    E = site_energies(ev, 2.0 * theta, off, x)
    (gt,) = torch.autograd.grad(E.sum(), theta, retain_graph=True)
    (gx,) = torch.autograd.grad(E.sum(), x, create_graph=True)
    (m,) = torch.autograd.grad(gx, theta, w, retain_graph=True)
    (gt2,) = torch.autograd.grad(E.sum(), theta, retain_graph=True)
    assert torch.equal(gt, gt2)
    assert torch.allclose(m, _mixed(site_energies(ev, 2.0 * theta, off, x), x, w, theta), rtol=1e-13)


def test_both_gradients_with_a_graph_of_their_own_that_is_not_kept():
    ev, off, theta, x, w = _setup()  # the parameters themselves: nothing behind them to keep
    want = _mixed(site_energies(ev, theta, off, x), x, w, theta)
    for inputs in ((theta, x), (x, theta)):
        E = site_energies(ev, theta, off, x)
        g = torch.autograd.grad(E.sum(), inputs, retain_graph=False, create_graph=True)
        (m,) = torch.autograd.grad(g[0] if inputs[0] is x else g[1], theta, w)
        assert torch.allclose(m, want, rtol=1e-13)
