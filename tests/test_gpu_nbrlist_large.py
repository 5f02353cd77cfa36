"""Neighbour lists near the entry points' limits (gpu): 2^31 - 48 entries, where
steps of 64 entries pass the largest 32-bit number."""
import numpy as np
import pytest
import torch

from acehip.atoms import NeighbourList

pytestmark = pytest.mark.gpu


def test_entries_up_to_the_limit(cuda):
    """A simple cubic lattice of 1 x 865 x 31,033 sites (periodic, so that sites
    meet their own images) with 80 neighbours each.  The reverse index is
    checked by its definition and the forces by their sum, at the end and at
    random; the gradients of the entries are whole numbers, so sums are exact."""
    if torch.cuda.mem_get_info()[0] < 170 << 30:
        pytest.skip("needs 170 GiB of device memory")
    dims, k = (1, 865, 31033), 80
    n, total = int(np.prod(dims)), 865 * 31033 * 80
    assert 2**31 - 64 < total < 2**31
    print(f"[gpu] {n} atoms, {total} entries", flush=True)
    i = torch.arange(n, device="cuda:0")
    pos = torch.stack([torch.zeros_like(i), i // dims[2], i % dims[2]]).double().contiguous()
    nl = NeighbourList(0)
    nl._alloc(total)
    nl.build(pos, np.diag(np.array(dims, dtype=float)), [1, 1, 1], 2.6)
    del i, pos
    assert nl.nnbr == total
    assert torch.equal(nl.offsets.long(), k * torch.arange(n + 1, device="cuda:0"))
    g = torch.Generator(device="cuda:0").manual_seed(1)
    m = torch.cat([torch.arange(total - 20000, total, device="cuda:0"),
                   torch.randint(0, total, (200000,), device="cuda:0", generator=g)])
    r, j = nl.rev[m].long(), nl.nbr_j[m]
    assert bool((nl.nbr_j[r] == m // k).all()) and bool((r // k == j).all())
    assert torch.equal(nl.shift[:, r], -nl.shift[:, m])
    dE = torch.empty((3, total), dtype=torch.float64, device="cuda:0")
    for d in range(3):
        dE[d].random_(-1000, 1000, generator=g)
    F = nl.forces(dE)
    atoms = torch.cat([torch.arange(n - 200, n, device="cuda:0"), torch.randint(0, n, (2000,), device="cuda:0")])
    e = (atoms[:, None] * k + torch.arange(k, device="cuda:0")).reshape(-1)
    want = (dE[:, e] - dE[:, nl.rev[e].long()]).view(3, len(atoms), k).sum(2)
    assert torch.equal(F[:, atoms], want)
    del dE, F, nl
    torch.cuda.empty_cache()
