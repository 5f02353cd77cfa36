"""Cotangents that are more than their memory (CPU, the oracle behind the
interface of the device evaluator): the row sums that the library computes
from a tensor's memory alone are left to torch for a forward-mode tangent, a
pending negation, a subclass, implicit zeros and batches, in the parameter
gradient and in the mixed second derivative."""
import ctypes as C

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from acehip.autograd import site_energies
from test_autograd_host import _case


class _RawRows:
    """The evaluator with row sums that read memory, as the device's do."""

    def __init__(self, ev):
        self.__dict__.update(ev=ev, raw=0)

    def __getattr__(self, name):
        return getattr(self.ev, name)

    def __setattr__(self, name, v):
        setattr(self.ev, name, v)

    def weighted_rows(self, w, B):
        self.__dict__["raw"] += 1
        w, B = w.contiguous(), B.contiguous()
        x, y = (np.ctypeslib.as_array(C.cast(t.data_ptr(), C.POINTER(C.c_double)), tuple(t.shape)) for t in (w, B))
        return torch.from_numpy(x @ y)


class _Twice(torch.Tensor):
    """A subclass whose product is not that of its memory."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs or {})
        return 2.0 * out.as_subclass(torch.Tensor) if func in (torch.Tensor.matmul, torch.Tensor.__matmul__) else out


@pytest.fixture
def case():
    ev, c, off, R = _case("Invariant", 3, 4)
    ev = _RawRows(ev)
    ct = torch.tensor(c, requires_grad=True)
    x = torch.tensor(R.T.copy(), requires_grad=True)
    rng = np.random.default_rng(0)
    E = site_energies(ev, ct, off, x)
    v, t = (torch.tensor(rng.normal(size=len(E))) for _ in range(2))
    (g,) = torch.autograd.grad(E, ct, v, retain_graph=True)
    assert ev.raw == 1  # a plain cotangent does go to the library
    return ev, ct, x, E, v, t, g


def _grad(E, ct, w):
    return torch.autograd.grad(E, ct, w, retain_graph=True)[0]


def test_forward_mode_tangent(case):
    ev, ct, x, E, v, t, g = case
    with fwAD.dual_level():
        primal, tangent = fwAD.unpack_dual(_grad(E, ct, fwAD.make_dual(v, t)))
        assert tangent is not None
    assert torch.allclose(primal, g, rtol=1e-13)
    assert torch.allclose(tangent, _grad(E, ct, t), rtol=1e-13)


def test_pending_negation_and_zeros(case):
    ev, ct, x, E, v, t, g = case
    assert torch.allclose(_grad(E, ct, torch._neg_view(v)), -g, rtol=1e-13)
    z = torch._efficientzerotensor(len(E), dtype=torch.float64)
    assert torch.equal(_grad(E, ct, z), torch.zeros_like(g))


def test_second_derivative(case):
    ev, ct, x, E, v, t, g = case
    w = torch.tensor(np.random.default_rng(1).normal(size=tuple(x.shape)))

    def mixed(cot):
        (gx,) = torch.autograd.grad(E, x, cot, create_graph=True)
        return torch.autograd.grad(gx, ct, w, retain_graph=True)[0]

    m = mixed(v)
    assert torch.allclose(mixed(torch._neg_view(v)), -m, rtol=1e-13)


def test_weighted_of_a_subclass(case):
    from acehip.autograd import _weighted
    ev, ct, x, E, v, t, g = case
    B = torch.tensor(np.random.default_rng(2).normal(size=(len(E), 5)))
    n = ev.raw
    assert torch.allclose(_weighted(ev, v.as_subclass(_Twice), B), 2.0 * (v @ B))
    assert ev.raw == n
