"""The slot programs (csrc/slots_host.hpp) run on the CPU against the A2B map
they stand for: the three components of E and dE/dA[k] from random pooled
values, whatever the split over workgroups.  The values need not come from
neighbours: both sides are polynomials in them.

Tolerance: both sides sum at most a few ten thousand products of four numbers
of order one in FP64, in another order; 1e-12 of the largest value is over 50
times the rounding that leaves."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from acehip import _lib, synth
from acehip.pack import Pack
from helpers import basis_for

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("args,kw", [((1, 4, 2), {}), ((2, 6, 3), {}), ((3, 6, 4), {}), ((3, 5, 3), {"species": 2}),
                                     ((3, 10, 5), {"species": 2})])
def test_slot_program(shim, args, kw):
    basis, T = basis_for(*args, prop="EuclideanVector", **kw)
    pk = Pack(T)
    assert pk.classed
    s, keep = _lib.make_pack(pk)
    rng = np.random.default_rng(5)
    c = synth.coefficients(len(basis), 5) * len(basis)
    npool = len(pk.pool)
    m = pk.pool[:, 3] > 0
    A = rng.normal(size=npool) + 1j * rng.normal(size=npool) * m
    # E_p = Re sum_AA c~_p prod A_f, and by reverse products dE_p = Re sum_k g[k, p] dA_k
    vals = np.asarray(pk.a2b_vals).reshape(-1, 3, 2) @ np.array([1.0, 1j])
    rows = np.repeat(np.arange(pk.nB), np.diff(pk.a2b_rowptr))
    ct = np.zeros((pk.nAA, 3), dtype=complex)
    np.add.at(ct, pk.a2b_cols, vals * c[rows][:, None])
    fid = np.asarray(pk.aspec_fid)
    k, cj = fid & 0x7fff, (fid & 0x8000) != 0
    full = np.asarray(pk.aspec_sgn) * np.where(cj, np.conj(A[k]), A[k])
    idx, orders = np.asarray(pk.iAA2iA).reshape(pk.nAA, -1), np.asarray(pk.orders)
    E0, G0 = np.zeros(3), np.zeros((npool, 3), dtype=complex)
    for o in range(int(orders.max()) + 1):
        sel = np.nonzero(orders == o)[0]
        x = full[idx[sel][:, :o]]
        E0 += np.sum(ct[sel] * np.prod(x, axis=1)[:, None], axis=0).real
        for q in range(o):
            d = np.prod(np.delete(x, q, axis=1), axis=1) * np.asarray(pk.aspec_sgn)[idx[sel][:, q]]
            v = ct[sel] * d[:, None]
            f = idx[sel][:, q]
            np.add.at(G0, k[f], np.where(cj[f][:, None], np.conj(v), v))
    scale = max(np.max(np.abs(E0)), np.max(np.abs(G0)))
    dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    Av = np.ascontiguousarray(np.stack([A.real, A.imag], -1))
    u, e0 = np.zeros((3, 3, 2)), np.zeros(3)
    assert shim.acehost_class(C.byref(s), dp(c), dp(u), dp(e0)) == 0
    u = u @ np.array([1.0, 1j])
    for forces in (1, 0):
        for P in (1, 3, 16):
            Q, G = np.zeros((3, 2)), np.zeros((npool, 3, 2))
            assert shim.acehost_slots(C.byref(s), dp(c), forces, P, dp(Av), dp(Q), dp(G)) == 0
            E = e0 + np.real((Q @ np.array([1.0, 1j])) @ u)
            assert np.max(np.abs(E - E0)) < 1e-12 * scale
            if forces:
                d = (G @ np.array([1.0, 1j])) @ u - G0
                # the real (m = 0) pooled values fix the real part only
                assert np.max(np.abs(np.where(m[:, None], d, d.real))) < 1e-12 * scale


def test_order_4_has_no_slot_form(shim):
    basis, T = basis_for(4, 5, 3, prop="EuclideanVector")
    s, keep = _lib.make_pack(Pack(T))
    z = np.zeros(65536)
    dp = z.ctypes.data_as(C.POINTER(C.c_double))
    c = synth.coefficients(len(basis), 5)
    assert shim.acehost_slots(C.byref(s), c.ctypes.data_as(C.POINTER(C.c_double)), 1, 1, dp, dp, dp) == 1
