"""The benchmark names and counts the product-DAG kernel that the library reports
(CPU): the segment kernel's counts are for the segment kernel alone, whatever
the basis."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import bench  # noqa: E402
import pytest  # noqa: E402
from acehip.pack import Pack  # noqa: E402
from helpers import basis_for  # noqa: E402


@pytest.mark.parametrize("args,kw", [((3, 6, 4), {}), ((4, 8, 4), {}), ((3, 6, 4), {"prop": "EuclideanVector"})])
def test_counts_follow_the_reported_kernel(args, kw):
    _, T = basis_for(*args, **kw)
    pk = Pack(T)
    seg = bench.executed_flops(pk, True, "segments", 0)
    assert seg > 0 and bench.lds_read_bytes(pk, True, "segments", 0) > 0
    assert bench.executed_flops(pk, True, "interpreter", 64) > 0
    assert bench.lds_read_bytes(pk, True, "interpreter", 64) is None
    for k in ("pairs", "slots"):
        assert bench.executed_flops(pk, True, k, 0) != seg
    assert bench.executed_flops(pk, True, "segments", 1) >= seg


def test_names():
    names = [bench.dag_kernel_name(k, t) for k, t in (("pairs", 0), ("slots", 0), ("slots", 1), ("segments", 0),
                                                      ("segments", 1), ("records", 0), ("interpreter", 32))]
    assert [n.split()[0] for n in names] == ["k_pairs", "k_slots", "k_slots", "k_dags", "k_dags", "k_dagr", "k_dag"]
    assert names[3] != names[4] and "32" in names[6]


def test_traffic_is_that_of_the_launch():
    whole, split = bench.dag_traffic("pairs", 100_000, 1, 0), bench.dag_traffic("pairs", 100_000, 2, 102)
    assert 0 < whole < split  # a split writes its shares of G
    for k, n, parts, tail in (("pairs", 100_000, 2, 0), ("pairs", 100_000, 3, 5), ("pairs", 50_000, 1, 0),
                              ("segments", 100_000, 1, 0)):
        assert bench.dag_traffic(k, n, parts, tail) is None
