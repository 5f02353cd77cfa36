"""The argument checks on the device (k_check, k_check_species): one bad offset
or species at the ends and in the middle of batches around a workgroup's 1,024
threads is refused with its message, a good batch of the same size after it is
not, and with offsets out of order no species is read."""
import numpy as np
import pytest
import torch

from acehip import synth
from acehip._lib import AceError
from acehip.evaluator import EnvBatch, HIPEvaluator
from helpers import basis_for, random_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nenv", [1, 2, 64, 65, 1024, 1025, 5000])
def test_device_checks(cuda, nenv):
    print(f"[gpu] device checks nenv {nenv}", flush=True)
    basis, _ = basis_for(2, 5, 3, species=2)
    ev = HIPEvaluator(basis, synth.coefficients(len(basis), 3), device=0)
    off, R, sp = random_batch(nenv, 5, nspecies=2)
    x = R.T.copy()
    E = ev.energy(EnvBatch(off, x, sp, device="cuda:0"))

    def refused(o, s, text):
        b = EnvBatch(off, x, sp, device="cuda:0")  # built from good offsets, changed on the device
        b.offsets.copy_(torch.as_tensor(o))
        b.species.copy_(torch.as_tensor(s))
        with pytest.raises(AceError, match=text):
            ev.energy(b)
        assert torch.equal(ev.energy(EnvBatch(off, x, sp, device="cuda:0")), E)

    for at in sorted({1, (nenv + 1) // 2, nenv - 1} & set(range(1, nenv))):
        o = off.copy()
        o[at] = off[at + 1] + 1
        refused(o, sp, "non-decreasing")
        refused(o, np.full_like(sp, 9), "non-decreasing")  # the offsets come first
    o = off.copy()
    o[0] = 1
    refused(o, sp, "start at 0")
    o = off.copy()
    o[nenv] = -1
    refused(o, sp, "start at 0 and be non-negative")
    for at in (0, len(sp) // 2, len(sp) - 1):
        for bad in (-1, 2):
            s = sp.copy()
            s[at] = bad
            refused(off, s, "species index out of range")
