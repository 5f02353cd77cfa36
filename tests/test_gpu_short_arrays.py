"""Offsets and species that end before what a batch claims are refused before
anything reads them, as the copies to the host that the checks once made were
(gpu)."""
import ctypes as C

import pytest
import torch

from acehip import synth
from acehip._lib import AceError, check
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch

pytestmark = pytest.mark.gpu


@pytest.fixture
def hip_block(cuda):
    """An allocation of its own, of exactly the bytes asked for."""
    torch.cuda.synchronize()
    hip = C.CDLL("libamdhip64.so")
    blocks = []

    def alloc(nbytes):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
        blocks.append(p)
        return p

    yield hip, alloc
    torch.cuda.synchronize()
    for p in blocks:
        assert hip.hipFree(p) == 0


def test_short_arrays_are_refused(cuda, hip_block):
    print("[gpu] offsets and species shorter than the batch claims", flush=True)
    hip, alloc = hip_block
    basis, _ = basis_for(2, 5, 3, species=2)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    off, R, sp = random_batch(40, 5, nspecies=2)
    b = EnvBatch(off, R.T.copy(), sp, device="cuda:0")
    E = ev.energy(b)
    out = torch.empty_like(E)

    def energy(nenv, offsets, species):
        torch.cuda.synchronize()
        check(ev.lib.ace_energy(ev.ctx, nenv, offsets, C.c_void_p(b.xyz.data_ptr()), species,
                                C.c_void_p(out.data_ptr()), ev._stream(None)))

    n = 1 << 20
    s = alloc(n)
    assert hip.hipMemset(s, 0, C.c_size_t(n)) == 0
    o = torch.tensor([0, 3, n, n + 1], dtype=torch.int32, device="cuda:0")
    with pytest.raises(AceError, match="species is shorter"):
        energy(3, C.c_void_p(o.data_ptr()), s)
    short = alloc(4 * n)
    with pytest.raises(AceError, match="env_offsets is shorter"):
        energy(n, short, s)
    # the good batch after it
    energy(40, C.c_void_p(b.offsets.data_ptr()), C.c_void_p(b.species.data_ptr()))
    torch.cuda.synchronize()
    assert torch.equal(out, E)
