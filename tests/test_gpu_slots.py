"""The slot kernel on the GPU against the oracle at the edges of its range:
tiles of 32 environments (one, a full one, one more, several), orders 1 to 3,
one and two species, more than 160 pooled values, energies alone, new
coefficients, and the allocation-free entry point bit for bit.  Tolerances are
those of the other parity tests (1e-12 for energies, 1e-10 for gradients, of
the largest value)."""
import numpy as np
import pytest
import torch

import ace_oracle as O
from acehip import synth
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("args,species,nenv", [((1, 4, 2), 0, 1), ((2, 6, 3), 0, 33), ((3, 6, 4), 0, 32),
                                               ((3, 5, 3), 2, 31), ((3, 7, 4), 0, 150), ((3, 9, 5), 2, 40)])
def test_slot_kernel(cuda, args, species, nenv):
    print(f"[gpu] slot kernel {args} species {species} nenv {nenv}", flush=True)
    basis, T = basis_for(*args, prop="EuclideanVector", species=species)
    c = synth.coefficients(len(basis), 3)
    off, R, sp = random_batch(nenv, 7, nspecies=species)
    ev = HIPEvaluator(basis, c, device=0)
    b = EnvBatch(off, R.T.copy(), sp, device="cuda:0")
    E0, g0 = O.energy(T, c, off, R, sp), O.grad_config(T, c, off, R, sp)
    for f in (1.0, -2.0):
        ev.set_params(f * np.asarray(c))
        E, dE = ev.energy_forces(b)
        E1 = ev.energy(b)
        En, dEn = ev.energy_forces_noalloc(b, torch.zeros_like(E), torch.zeros_like(dE))
        torch.cuda.synchronize()
        assert torch.equal(E, En) and torch.equal(dE, dEn)
        assert rel_err(E.cpu().numpy(), f * E0) < 1e-12 and rel_err(E1.cpu().numpy(), f * E0) < 1e-12
        g = dE.cpu().numpy().reshape(3, 3, -1).transpose(2, 0, 1)
        assert rel_err(g, f * g0) < 1e-10
