"""The device buffers' rule (csrc/grow_buf.hpp) on the CPU: a block that a
captured call used outlives every later call, whichever batch needs more room,
and no other replaced block does; all are given back with the buffer."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    return C.CDLL(str(so))


# (elements, captured) of each call, and the blocks that are alive after them
CASES = [
    # G of 8,192 and then of 5,000 and 6,000 order-4 environments (KB), whose
    # splits need more room than the larger batch's
    ([(21, 0), (21, 1), (45, 0), (67, 0)], 2),
    ([(21, 0), (45, 0), (67, 0)], 1),  # nothing captured: one block
    ([(21, 1), (45, 1), (45, 0), (67, 0), (80, 0)], 3),
    ([(45, 1), (21, 0), (21, 1)], 1),  # room enough: no second block
]


@pytest.mark.parametrize("calls,alive", CASES)
def test_blocks_of_captured_calls_are_kept(shim, calls, alive):
    sizes = np.array([1000 * c[0] for c in calls], dtype=np.int64)
    cap = np.array([c[1] for c in calls], dtype=np.int32)
    graphs, blocks, left = C.c_int(), C.c_int(), C.c_int()
    ok = shim.acehost_grow_buf(sizes.ctypes.data_as(C.c_void_p), cap.ctypes.data_as(C.c_void_p), len(calls),
                               C.byref(graphs), C.byref(blocks), C.byref(left))
    assert ok == graphs.value == sum(c[1] for c in calls) and blocks.value == alive and left.value == 0
