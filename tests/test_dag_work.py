"""What the pair and the slot kernel execute per environment
(ace_last_dag_work's counts) on the CPU: against the hardware's counter of FP64
operations at the headline workload, and against the programs' own sizes, of
which the counts are sums (a column 19 operations and 32 bytes or fewer per
lane, a step 76 and 64; two lanes have an environment)."""
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
def work(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    lib = C.CDLL(str(so))

    def run(args, kw, forces):
        _, T = basis_for(*args, **kw)
        s, keep = _lib.make_pack(Pack(T))
        out = np.zeros(5)
        assert lib.acehost_dag_work(C.byref(s), int(forces), out.ctypes.data_as(C.c_void_p)) == 0
        return out

    return run


def test_headline_workload_as_counted(work):
    # SQ_INSTS_VALU_FLOPS_FP64 of a launch of whole tiles, 100,000 environments: 528.1 M x 64 lanes
    assert abs(work((4, 12, 6), {}, True)[0] / (528.1e6 * 64 / 100_000) - 1.0) < 1e-3


@pytest.mark.parametrize("forces", [True, False])
@pytest.mark.parametrize("args", [(3, 6, 4), (4, 8, 4), (5, 6, 3)])
def test_pairs(work, args, forces):
    flops, lds, cols, panels, virt = work(args, {}, forces)
    rest = flops - 2 * (19 * cols + 8 * (8 if forces else 5) * panels + 3 * virt)
    # with forces, each factor of a product of its own takes four more
    assert rest == (2 * 2 * 4 * virt if forces else 0)
    assert 2 * 16 * cols < lds < 2 * (32 * cols + 256 * panels + 32 * 200 + 96 * virt)


@pytest.mark.parametrize("forces", [True, False])
@pytest.mark.parametrize("args", [(3, 6, 4), (3, 10, 5)])
def test_slots(work, args, forces):
    flops, lds, steps, pieces, slots = work(args, {"prop": "EuclideanVector"}, forces)
    rows = (flops - 2 * (76 * steps + (48 * pieces if forces else 0))) / (2 * (9 if forces else 8))
    assert rows == (slots if forces else round(rows)) and 0 < rows <= 4 * pieces
    assert lds == 2 * (64 * steps + 16 * rows)
