"""A captured call keeps its scratch (gpu), of a context and of a neighbour
list: after eager calls on smaller batches
that need more room (their tiles are split further), each replay still gives
the eager result, bit for bit, with other memory handed out in between."""
import numpy as np
import pytest
import torch

from acehip import synth
from acehip.atoms import NeighbourList
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for

pytestmark = pytest.mark.gpu


def _capture(run):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run()
    return g


@pytest.mark.parametrize("args,kw,wid,captured,others", [
    ((4, 12, 6), {}, 2, 8192, (5000, 6000)),  # the pair kernel's G shares
    ((3, 10, 5), {"prop": "EuclideanVector", "species": 2}, 4, 16384, (8193,)),  # the slot kernel's energy shares
], ids=["pairs", "slots"])
def test_replay_after_smaller_eager_batches(cuda, args, kw, wid, captured, others):
    print(f"[gpu] capture {captured} envs, evaluate {others}, replay", flush=True)
    basis, _ = basis_for(*args, **kw)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), wid), device=0, waves=16)
    ev.set_validation(False)

    def batch(n, seed):
        off, R, sp = synth.workload_envs(wid, nenv=n, seed=seed)
        return EnvBatch(off, R.T.copy(), sp, device="cuda:0")

    b = batch(captured, 11)
    E0, dE0 = ev.energy_forces(b)
    E, dE = torch.empty_like(E0), torch.empty_like(dE0)
    g = _capture(lambda: ev.energy_forces(b, E, dE))
    for i, n in enumerate(others + (None,) * 2):
        if n is not None:
            ev.energy_forces(batch(n, 20 + i))
        hog = [torch.full((1 << 24,), float("nan"), dtype=torch.float64, device="cuda:0") for _ in range(2)]
        E.zero_()
        dE.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(E, E0) and torch.equal(dE, dE0), n
        assert all(bool(h.isnan().all()) for h in hog)
        del hog


def test_replay_of_forces_after_fewer_atoms(cuda):
    """The virial's shares: 32,768 atoms take more workgroups than 40,000."""
    print("[gpu] capture the forces of 40,000 atoms, then 32,768 on the same list", flush=True)
    rng = np.random.default_rng(3)

    def listed(n):
        a = (8.0 * n) ** (1.0 / 3.0)  # about four neighbours within 2
        nl = NeighbourList(0).build(rng.uniform(0.0, a, size=(n, 3)), a * np.eye(3), [1, 1, 1], 2.0)
        return nl, torch.tensor(rng.normal(size=(3, nl.nnbr)), device="cuda:0")

    nl, g = listed(40000)
    few, gf = listed(32768)
    few.h, own = nl.h, few.h  # the other list's arrays through the same handle
    F0, W0 = nl.forces(g, virial=True)
    F, W = torch.empty_like(F0), torch.empty_like(W0)
    graph = _capture(lambda: nl._forces(g, F, W))
    try:
        for rep in range(4):
            few.forces(gf, virial=True)
            hog = torch.full((1 << 20,), float("nan"), dtype=torch.float64, device="cuda:0")
            F.zero_()
            W.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(F, F0) and torch.equal(W, W0), rep
            assert bool(hog.isnan().all())
    finally:
        few.h = own


@pytest.mark.parametrize("args,kw,wid,sizes", [
    ((4, 12, 6), {}, 2, (1500, 9000)),
    # the slot kernel's energies over more workgroups than its forces: 6 against 3, 7 against 6
    ((3, 10, 5), {"prop": "EuclideanVector"}, 4, (64, 700)),
    ((3, 10, 5), {"prop": "EuclideanVector", "species": 2}, 4, (3300,)),
], ids=["pairs", "slots", "slots2"])
def test_energies_captured_after_forces(cuda, args, kw, wid, sizes):
    """One eager call on the batch precedes a capture, in either mode: the call
    with forces also makes the room for the energies alone."""
    basis, _ = basis_for(*args, **kw)
    c = synth.coefficients(len(basis), wid)
    for n in sizes:
        print(f"[gpu] energies of {n} envs captured after an eager call with forces", flush=True)
        off, R, sp = synth.workload_envs(wid, nenv=n, seed=31)
        b = EnvBatch(off, R.T.copy(), sp if kw.get("species") else None, device="cuda:0")
        E0 = HIPEvaluator(basis, c, device=0, waves=16).energy(b)
        ev = HIPEvaluator(basis, c, device=0, waves=16)
        ev.set_validation(False)
        E = torch.empty_like(E0)
        ev.energy_forces(b)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            ev.energy(b, E)
        for rep in range(3):
            E.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(E, E0), (n, rep)
            ev.energy_forces(b)
