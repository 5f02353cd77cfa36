"""The choice of tail tiles (csrc/tail_host.hpp) on the CPU: the same number as
a dispatch of one workgroup after another, and cheap enough for the first call
of a tile count (a heap of the units took 1 to 2.5 ms, as long as the call)."""
import ctypes as C
import heapq
import os
import subprocess
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    so = tmp_path_factory.mktemp("shim") / "libacehost.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-o", str(so),
                    os.path.join(ROOT, "ace.jl_amd", "csrc", "pack_host_check.cpp")], check=True)
    f = C.CDLL(str(so)).acehost_choose_tail
    f.restype = C.c_int64
    f.argtypes = [C.c_int64, C.c_int, C.c_int, C.c_double, C.c_double]
    return f


def dispatched(ntile, P, ncu, d, dh):
    ms = []
    for nhi in range(min(ntile, ncu) + 1):
        full, rest = divmod((ntile - nhi) * P, ncu)
        h = [(full + (i < rest)) * d for i in range(ncu)]
        heapq.heapify(h)
        for _ in range(nhi * (P + 1)):
            heapq.heapreplace(h, h[0] + dh)
        ms.append(max(h))
    ties = [n for n, m in enumerate(ms) if m <= min(ms) * (1.0 + 1e-9)]
    return ties[len(ties) // 2]


def test_same_as_one_after_another(choose):
    rng = np.random.default_rng(4)
    for i in range(60):
        ncu, P, ntile = int(rng.integers(1, 40)), int(rng.integers(2, 9)), int(rng.integers(1, 300))
        work = rng.uniform(1e5, 1e6)
        d, dh = work / P + 17000.0, work / (P + 1) * rng.uniform(1.0, 1.1) + 17000.0
        if i % 2:
            d, dh = 1.0 / P, 1.08 / (P + 1)
        assert choose(ntile, P, ncu, d, dh) == dispatched(ntile, P, ncu, d, dh), (ntile, P, ncu)


def test_cost(choose):
    t = time.perf_counter()
    for ntile in range(400, 700):
        choose(ntile, 4, 256, 67000.0, 57000.0)
    assert time.perf_counter() - t < 0.15  # 0.5 ms each; measured 0.004
