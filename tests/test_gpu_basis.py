"""Fused basis values and their directional derivative on the GPU against the
oracle at the edges of the kernel's range: tiles of 32 environments (one, a
full one, one more, several), orders 1 to 4, one and two species, pooled
values up to the limit of two staged tiles (160) and past it.  Tolerances are
those of the other parity tests (1e-12 for values, 1e-10 for derivatives)."""
import numpy as np
import pytest
import torch

import ace_oracle as O
from acehip import synth
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("args,species,nenv", [((1, 4, 2), 0, 1), ((2, 6, 3), 0, 33), ((3, 6, 4), 0, 32),
                                               ((4, 8, 4), 0, 97), ((3, 6, 3), 2, 31), ((2, 13, 6), 0, 40),
                                               ((2, 16, 7), 0, 5), ((4, 10, 5), 0, 700)])
def test_basis_values(cuda, args, species, nenv):
    print(f"[gpu] basis values {args} species {species} nenv {nenv}", flush=True)
    basis, T = basis_for(*args, species=species)
    off, R, sp = random_batch(nenv, 9, nspecies=species)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    b = EnvBatch(off, R.T.copy(), sp, device="cuda:0")
    w = np.random.default_rng(4).normal(size=R.shape)
    B = ev.basis_B(b).cpu().numpy()
    D = ev.adjoint_EVAL_D(b, torch.as_tensor(w.T.copy())).cpu().numpy()
    assert rel_err(B, O.eval_B(T, O.eval_AA(T, O.eval_A(T, off, R, sp)))) < 1e-12
    # the oracle's derivative one environment at a time: the first and the last ones
    es = sorted(set(range(min(nenv, 40))) | set(range(max(0, nenv - 9), nenv)))
    ref = [O.adjoint_EVAL_D(T, None, off[e:e + 2] - off[e], R[off[e]:off[e + 1]], w[off[e]:off[e + 1]],
                            None if sp is None else sp[off[e]:off[e + 1]]) for e in es]
    assert rel_err(D[es], np.stack(ref).reshape(len(es), -1)) < 1e-10


@pytest.mark.parametrize("nrow,ncol", [(0, 3), (1, 1), (7, 255), (8, 257), (65, 64), (2003, 97), (50001, 2), (333, 3235)])
def test_weighted_rows(cuda, nrow, ncol):
    """Shares of rows and columns past a workgroup's 256; sums of at most 50,001
    products of numbers of order one in FP64: 1e-12 of the largest possible sum."""
    print(f"[gpu] weighted rows {nrow} x {ncol}", flush=True)
    basis, _ = basis_for(1, 4, 2)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    rng = np.random.default_rng(nrow)
    w, B = rng.uniform(-1, 1, nrow), rng.uniform(-1, 1, (nrow, ncol))
    got = ev.weighted_rows(torch.as_tensor(w).cuda(), torch.as_tensor(B).cuda()).cpu().numpy()
    assert got.shape == (ncol,) and np.max(np.abs(got - w @ B)) <= 1e-12 * max(1, nrow)


def test_batched_cotangents(cuda):
    """A batch of cotangents (legacy vmap tensors, which have no storage) takes
    torch's product, single ones the kernel: the same gradients."""
    from acehip.autograd import site_energies
    basis, _ = basis_for(2, 5, 3)
    c = synth.coefficients(len(basis), 3)
    ev = HIPEvaluator(basis, c, device=0)
    off, R, _ = random_batch(5, 8)
    ct = torch.as_tensor(c, device="cuda").requires_grad_(True)
    E = site_energies(ev, ct, off, torch.as_tensor(R.T.copy(), device="cuda"))
    eye = torch.eye(5, dtype=torch.float64, device="cuda")
    (g,) = torch.autograd.grad(E, ct, eye, is_grads_batched=True, retain_graph=True)
    one = torch.stack([torch.autograd.grad(E, ct, v, retain_graph=True)[0] for v in eye])
    assert torch.allclose(g, one, rtol=1e-12, atol=1e-14)


@pytest.mark.parametrize("args,kw", [((1, 4, 2), {}), ((3, 6, 4), {}), ((4, 8, 4), {}), ((5, 5, 3), {}),
                                     ((3, 5, 3), {"prop": "EuclideanVector", "species": 2})])
def test_basis_gradients(cuda, args, kw):
    """Basis gradients by adjoint weights: fewer functions than a wave and several
    windows of 256, entries of four and of eight factors, merged (Invariant) and
    not (vector); against the oracle (1e-10 of the largest value)."""
    print(f"[gpu] basis gradients {args} {kw}", flush=True)
    basis, T = basis_for(*args, **kw)
    off, R, sp = random_batch(5, 3, nspecies=kw.get("species", 0))
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    dB = ev.basis_dB(EnvBatch(off, R.T.copy(), sp, device="cuda:0")).cpu().numpy()
    _, dAA = O.eval_AA_dAA(T, off, R, sp)
    ref = O.eval_dB(T, dAA)
    assert dB.size == ref.size
    assert rel_err(dB.reshape(ref.shape), ref) < 1e-10
