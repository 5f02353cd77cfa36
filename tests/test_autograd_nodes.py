"""Which evaluations a gradient of the site energies runs (CPU, the oracle
behind the interface of the device evaluator): positions alone do not evaluate
the basis, parameters alone not the pullback; the energies may be written to in
place; batched cotangents give the gradients of each."""
import numpy as np
import pytest
import torch

from acehip.autograd import site_energies
from test_autograd_host import _case


class _Counting:
    def __init__(self, ev):
        self.__dict__["ev"] = ev
        self.__dict__["calls"] = []

    def __getattr__(self, name):
        v = getattr(self.ev, name)
        if name in ("basis_B", "adjoint_EVAL_D", "energy_forces"):
            self.calls.append(name)
        return v

    def __setattr__(self, name, v):
        setattr(self.ev, name, v)


@pytest.mark.parametrize("prop", ["Invariant", "EuclideanVector"])
def test_gradients_run_only_what_they_need(prop):
    ev, c, off, R = _case(prop, 3, 4)
    ev = _Counting(ev)
    ct = torch.tensor(c, requires_grad=True)
    x = torch.tensor(R.T.copy(), requires_grad=True)
    E = site_energies(ev, ct, off, x)
    del ev.calls[:]
    (gx,) = torch.autograd.grad(E.sum(), x, retain_graph=True)
    assert ev.calls == []
    (gc,) = torch.autograd.grad(E.sum(), ct, retain_graph=True)
    assert ev.calls == ["basis_B"]
    both = torch.autograd.grad(E.sum(), (x, ct), retain_graph=True)
    assert torch.equal(both[0], gx) and torch.equal(both[1], gc)
    if prop == "Invariant":  # a batch of cotangents (the vector contraction has no batching rule)
        (gb,) = torch.autograd.grad(E, ct, torch.eye(len(E), dtype=torch.float64), is_grads_batched=True,
                                    retain_graph=True)
        assert torch.allclose(gb.sum(0), gc, rtol=1e-12, atol=1e-13)
    # a fresh tensor, and parameters that changed since are noticed
    E.mul_(2.0)
    (g2,) = torch.autograd.grad(E.sum(), x, retain_graph=True)
    assert torch.allclose(g2, 2.0 * gx)
    with torch.no_grad():
        ct.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(E.sum(), x)
