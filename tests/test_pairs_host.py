"""The pair programs (csrc/pairs_host.hpp) run on the CPU against the
polynomials they stand for: energy and G[k] from random pooled values, and
the schedule's rule that panels of one turn share no target.  The values need
not come from neighbours: both sides are polynomials in them.

Tolerance: both sides sum at most a few ten thousand products of four
numbers of order one in FP64, in another order; 1e-12 of the largest value is
over 50 times the rounding that leaves."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from acehip import _lib, synth
from acehip import programs as P
from acehip.pack import Pack
from helpers import basis_for

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    return C.CDLL(str(so))


def direct(pk, ct, A):
    """E (without the constant) and G of the energy polynomial at A."""
    X = lambda f: np.conj(A[f >> 1]) if f & 1 else A[f >> 1]  # noqa: E731
    E, G = 0.0, np.zeros(len(A), dtype=complex)
    for mono, terms in pk.poly.items():
        co = float(np.real(P.eval_terms(terms, ct)))
        x = [X(f) for f in mono]
        E += co * np.prod(x).real
        for i, f in enumerate(mono):
            d = co * np.prod(x[:i] + x[i + 1:])
            G[f >> 1] += np.conj(d) if f & 1 else d
    return E, G


@pytest.mark.parametrize("args,kw", [((1, 4, 2), {}), ((2, 5, 3), {}), ((3, 6, 4), {}), ((4, 8, 4), {}),
                                     ((4, 12, 6), {}), ((2, 13, 5), {}), ((3, 6, 3), {"species": 2}),
                                     # monomials brought to four factors first
                                     ((5, 6, 3), {}), ((5, 5, 3), {"species": 2}), ((6, 6, 3), {}), ((7, 5, 2), {})])
def test_pair_program(shim, args, kw):
    basis, T = basis_for(*args, **kw)
    pk = Pack(T)
    s, keep = _lib.make_pack(pk)
    rng = np.random.default_rng(5)
    c = synth.coefficients(len(basis), 5) * len(basis)
    A = rng.normal(size=len(pk.pool)) + 1j * rng.normal(size=len(pk.pool)) * (pk.pool[:, 3] > 0)
    ct = np.zeros(pk.nAA)
    rows = np.repeat(np.arange(pk.nB), np.diff(pk.a2b_rowptr))
    np.add.at(ct, pk.a2b_cols, pk.a2b_vals * c[rows])
    E0, G0 = direct(pk, ct, A)
    E0 += float(np.sum(ct[pk.orders == 0]))
    scale = max(abs(E0), np.max(np.abs(G0)))
    dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    Av = np.ascontiguousarray(np.stack([A.real, A.imag], -1))
    for forces in (1, 0):
        for parts in (1, 2, 3, 9):
            E, G = np.zeros(1), np.zeros((len(A), 2))
            assert shim.acehost_pairs(C.byref(s), dp(c), forces, parts, dp(Av), dp(E), dp(G)) == 0
            assert abs(E[0] - E0) < 1e-12 * scale
            if forces:
                d = G[:, 0] + 1j * G[:, 1] - G0
                # the real (m = 0) pooled values fix the real part only
                assert np.max(np.abs(np.where(pk.pool[:, 3] > 0, d, d.real))) < 1e-12 * scale
