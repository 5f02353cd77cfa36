"""The pair kernel on the GPU against the oracle at the edges of its range:
tiles of 32 environments (one, a full one, one more), few and many pooled
values up to its limit of 159 and past it (another kernel), one and two
species, an order-3 batch past one tile per compute unit (another kernel),
orders 5 to 7, and every split of a tile over workgroups, whose G shares the force
kernels add up.  Tolerances are those of the other parity tests (1e-12 for
energies, 1e-10 for gradients, of the largest value); splits only change the
order of a few sums, 1e-13."""
import numpy as np
import pytest
import torch

import ace_oracle as O
from acehip import synth
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("args,species,nenv", [((3, 4, 2), 0, 33), ((4, 5, 3), 0, 1), ((3, 6, 4), 0, 32),
                                               ((3, 13, 5), 0, 9), ((2, 13, 6), 0, 40), ((3, 6, 3), 2, 31),
                                               ((4, 8, 4), 0, 70), ((3, 6, 4), 0, 8193),
                                               # products of their own behind the pooled values
                                               ((5, 6, 3), 0, 33), ((5, 5, 3), 2, 40), ((7, 5, 2), 0, 65)])
def test_pair_kernel(cuda, args, species, nenv):
    print(f"[gpu] pair kernel {args} species {species} nenv {nenv}", flush=True)
    basis, T = basis_for(*args, species=species)
    c = synth.coefficients(len(basis), 3)
    off, R, sp = random_batch(nenv, 7, nspecies=species) if nenv < 1000 else synth.random_envs(nenv, "fixed5", 7)
    ev = HIPEvaluator(basis, c, device=0)
    b = EnvBatch(off, R.T.copy(), sp, device="cuda:0")
    n = min(nenv, 70)  # the oracle's share
    o, Rn, sn = off[:n + 1], R[:off[n]], None if sp is None else sp[:off[n]]
    E0, g0 = O.energy(T, c, o, Rn, sn), O.grad_config(T, c, o, Rn, sn)
    first = None
    for parts, tail in ((0, -1), (1, -1), (2, 0), (2, 1), (3, 1), (4, 0)):
        ev.set_parts(parts)
        ev.set_tail_parts(tail)
        E, dE = ev.energy_forces(b)
        E1 = ev.energy(b)
        torch.cuda.synchronize()
        E, dE, E1 = E.cpu().numpy()[:n], dE.cpu().numpy().T[:off[n]], E1.cpu().numpy()[:n]
        assert rel_err(E, E0) < 1e-12 and rel_err(E1, E0) < 1e-12, (parts, tail)
        assert rel_err(dE, g0) < 1e-10, (parts, tail)
        if parts:
            P, nt, kern = ev.last_dag_shape()
            assert kern == (0 if ev.npool <= 160 else 1) and (P, nt) == (parts, max(0, tail))
        first = first or (E, dE)
        assert rel_err(E, first[0]) < 1e-13 and rel_err(dE, first[1]) < 1e-13
    # new coefficients reach the programs
    ev.set_parts(0)
    ev.set_tail_parts(-1)
    ev.set_params(-2.0 * np.asarray(c))
    E, dE = ev.energy_forces(b)
    assert rel_err(E.cpu().numpy()[:n], -2.0 * E0) < 1e-12
    assert rel_err(dE.cpu().numpy().T[:off[n]], -2.0 * g0) < 1e-10


@pytest.mark.parametrize("rounds,extra", [(1, 1), (4, 0), (4, 5)])
def test_whole_tiles_or_a_split(cuda, rounds, extra):
    """More tiles than compute units: whole tiles where their rounds are full,
    a split or whole tiles past that, the same sums either way (1e-13)."""
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    nenv = 32 * ncu * rounds + extra
    print(f"[gpu] pair kernel whole tiles or a split, {nenv} environments", flush=True)
    basis, _ = basis_for(4, 5, 3)
    off, R, sp = synth.random_envs(nenv, "fixed5", 11)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    b = EnvBatch(off, R.T.copy(), sp, device="cuda:0")
    E, dE = ev.energy_forces(b)
    if extra == 0:
        assert ev.last_dag_shape()[:2] == (1, 0)
    E, dE = E.cpu().numpy(), dE.cpu().numpy()
    for parts in (1, 2):
        ev.set_parts(parts)
        E1, dE1 = ev.energy_forces(b)
        assert rel_err(E, E1.cpu().numpy()) < 1e-13 and rel_err(dE, dE1.cpu().numpy()) < 1e-13
