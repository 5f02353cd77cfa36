"""The records of the fused basis values (csrc/basis_host.hpp) run on the CPU
against the A2B table they come from, values and directional derivatives, and
every row written once however the rows are split.

Tolerance: a row sums at most a few hundred products of four numbers of order
one in FP64, in another order; 1e-13 of the largest value is over 50 times
the rounding that leaves."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from acehip import _lib
from acehip.pack import Pack
from helpers import basis_for

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("args,kw", [((1, 4, 2), {}), ((2, 5, 3), {}), ((3, 6, 4), {}), ((4, 8, 4), {}),
                                     ((4, 12, 6), {}), ((3, 6, 3), {"species": 2})])
def test_basis_records(shim, args, kw):
    basis, T = basis_for(*args, **kw)
    pk = Pack(T)
    s, keep = _lib.make_pack(pk)
    rng = np.random.default_rng(7)
    m = pk.pool[:, 3] > 0
    A, W = (rng.normal(size=len(m)) + 1j * rng.normal(size=len(m)) * m for _ in range(2))
    fid = np.asarray(pk.aspec_fid)
    full = lambda X: np.asarray(pk.aspec_sgn) * np.where(fid & 0x8000, np.conj(X[fid & 0x7fff]), X[fid & 0x7fff])  # noqa: E731
    a, w = full(A), full(W)
    idx = np.asarray(pk.iAA2iA).reshape(pk.nAA, -1)
    x, dx = np.ones(pk.nAA, dtype=complex), np.zeros(pk.nAA, dtype=complex)
    for q in range(idx.shape[1]):
        on = np.asarray(pk.orders) > q
        i = np.where(on, idx[:, q], 0)
        dx = np.where(on, dx * a[i] + x * w[i], dx)
        x = np.where(on, x * a[i], x)
    rows = np.repeat(np.arange(pk.nB), np.diff(pk.a2b_rowptr))
    B0, D0 = np.zeros(pk.nB), np.zeros(pk.nB)
    np.add.at(B0, rows, pk.a2b_vals * x[pk.a2b_cols].real)
    np.add.at(D0, rows, pk.a2b_vals * dx[pk.a2b_cols].real)
    dp = lambda v: v.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    Av, Wv = (np.ascontiguousarray(np.stack([v.real, v.imag], -1)) for v in (A, W))
    for nchunk in (1, 3, 48):
        B, D = np.zeros(pk.nB), np.zeros(pk.nB)
        assert shim.acehost_bv(C.byref(s), nchunk, dp(Av), dp(Wv), dp(B), dp(D)) == 0
        assert np.max(np.abs(B - B0)) < 1e-13 * np.max(np.abs(B0))
        assert np.max(np.abs(D - D0)) < 1e-13 * np.max(np.abs(D0))
