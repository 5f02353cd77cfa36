"""The library reports the product-DAG kernel that it launched (gpu): at the
edges of each dispatch rule, with forces and for energies alone.  The
benchmark's line names and counts what is reported."""
import pytest
import torch

from acehip import synth
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch

pytestmark = pytest.mark.gpu

VEC = {"prop": "EuclideanVector"}
# basis, environments, kernel with forces, kernel of the energies alone
CASES = [
    ((4, 8, 4), {}, 5, "pairs", "pairs"),
    ((4, 8, 4), {}, 9000, "pairs", "pairs"),
    ((3, 6, 4), {}, 1000, "pairs", "pairs"),       # order 3 up to one tile per compute unit
    ((3, 6, 4), {}, 9000, "segments", "pairs"),
    ((2, 5, 3), {}, 100, "segments", "segments"),
    ((5, 6, 3), {}, 100, "pairs", "pairs"),
    ((8, 5, 2), {}, 100, "segments", "segments"),  # no pair form above order 7
    ((3, 6, 4), VEC, 100, "slots", "segments"),
    ((2, 5, 3), VEC, 100, "segments", "segments"),
]


def _run(ev, b):
    got = []
    for run in (ev.energy_forces, ev.energy):
        run(b)
        got.append(ev.last_dag_kernel())
        work = ev.last_dag_work()  # counted by the library for the kernels with programs of their own
        assert (work is not None) == (got[-1] in ("pairs", "slots")) and (work is None or min(work) > 0)
    return tuple(got)


@pytest.mark.parametrize("args,kw,nenv,forces,energy", CASES)
def test_reported_kernel(cuda, args, kw, nenv, forces, energy):
    print(f"[gpu] kernel of {args} {kw} {nenv} envs", flush=True)
    basis, _ = basis_for(*args, **kw)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 1), device=0)
    assert ev.last_dag_kernel() is None
    off, R, _ = random_batch(nenv, 4)
    b = EnvBatch(off, R.T.copy(), None, device="cuda:0")
    assert _run(ev, b) == (forces, energy)
    ev.set_kernel(1)
    assert _run(ev, b) == ("interpreter", "interpreter")
    if args[0] <= 4:
        ev.set_kernel(2)
        assert _run(ev, b) == ("records", "records")
    ev.set_kernel(0)
    ev.set_parts(2)  # a split that the caller set: the slot kernel leaves the call
    assert _run(ev, b) == tuple("segments" if k == "slots" else k for k in (forces, energy))
    ev.set_parts(0)
    assert _run(ev, b) == (forces, energy)
    torch.cuda.synchronize()
