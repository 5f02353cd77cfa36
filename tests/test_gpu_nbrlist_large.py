"""Neighbour lists near the entry points' limits (gpu): 2^31 - 48 entries, where
steps of 64 entries pass the largest 32-bit number, and more than 2^26 atoms,
whose waves are more threads than one launch takes; and many positions that
are not finite."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from acehip._lib import AceError, check
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


def test_more_atoms_than_one_launch_takes(cuda):
    """2^26 sites of a cubic lattice of spacing 1 without neighbours within 0.9,
    and five atoms half-way between two of them."""
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GiB of device memory")
    n0, dims = 1 << 26, (512, 512, 256)
    print(f"[gpu] {n0 + 5} atoms", flush=True)
    i = torch.arange(n0, device="cuda:0")
    site = torch.stack([i // (dims[1] * dims[2]), i // dims[2] % dims[1], i % dims[2]]).double()
    near = torch.tensor([0, 12345678, n0 // 2, n0 - 1000, n0 - 1], device="cuda:0")
    step = torch.tensor([[0.5], [0.0], [0.0]], dtype=torch.float64, device="cuda:0")
    pos = torch.cat([site, site[:, near] + step], 1).contiguous()
    del i, site
    nl = NeighbourList(0).build(pos, np.diag(np.array(dims, dtype=float)), [1, 1, 1], 0.9)
    other = (near + dims[1] * dims[2]) % n0  # the next site along x
    assert nl.nnbr == 20
    cnt = torch.zeros(n0 + 5, dtype=torch.int64, device="cuda:0")
    cnt[n0:] = 2
    for s in (near, other):
        cnt[s] += 1
    assert torch.equal((nl.offsets[1:] - nl.offsets[:-1]).long(), cnt)
    i = torch.repeat_interleave(torch.arange(n0 + 5, device="cuda:0"), cnt)
    assert torch.equal(nl.nbr_j[-10:].long().view(5, 2).sort(1).values, torch.stack([near, other], 1).sort(1).values)
    rev = nl.rev.long()
    assert torch.equal(nl.nbr_j[rev].long(), i) and torch.equal(nl.shift[:, rev], -nl.shift)
    assert torch.equal(nl.xyz.abs()[0], torch.full((20,), 0.5, dtype=torch.float64, device="cuda:0"))
    assert not nl.xyz[1:].any()
    nl.update(pos + 0.25 * torch.arange(n0 + 5, device="cuda:0").eq(n0 + 4))
    assert torch.equal(nl.xyz[:, -2:].abs().sum(0).sort().values,
                       torch.tensor([0.75, 1.25], dtype=torch.float64, device="cuda:0"))
    del pos, cnt, i, nl
    torch.cuda.empty_cache()


def test_update_of_more_atoms_than_one_launch_takes(cuda):
    """2^28 + 32 atoms at 16 threads each; the last has the only two entries."""
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GiB of device memory")
    n = (1 << 28) + 32
    print(f"[gpu] update of {n} atoms", flush=True)
    pos = torch.zeros((3, n), dtype=torch.float64, device="cuda:0")
    pos[:, 5] = 1.0
    pos[0, n - 1] = 4.0
    off = torch.zeros(n + 1, dtype=torch.int32, device="cuda:0")
    off[n] = 2
    nl = NeighbourList(0)
    j = torch.tensor([5, 7], dtype=torch.int32, device="cuda:0")
    shift = torch.tensor([[0, 1], [0, 0], [0, 0]], dtype=torch.int32, device="cuda:0")
    xyz = torch.full((3, 2), float("nan"), dtype=torch.float64, device="cuda:0")
    cell = (C.c_double * 9)(10.0, 0, 0, 0, 10.0, 0, 0, 0, 10.0)
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    check(nl.lib.ace_nbrlist_update(nl.h, n, p(pos), cell, 2, p(off), p(j), p(shift), p(xyz), nl._stream(None)))
    assert torch.equal(xyz, torch.tensor([[-3.0, 6.0], [1.0, 0.0], [1.0, 0.0]], dtype=torch.float64, device="cuda:0"))
    del pos, off, nl
    torch.cuda.empty_cache()


def test_positions_gone_bad_are_refused_at_once(cuda):
    """They all fall into one bin, where a search would compare each of the
    three million with every other (over ten seconds)."""
    n = 3_000_000
    print(f"[gpu] {n} positions that are not numbers", flush=True)
    nl = NeighbourList(0)
    cell = 150.0 * np.eye(3)
    for value, text in ((float("nan"), "finite"), (1e12, "too far outside")):
        bad = torch.full((3, n), value, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        t = time.perf_counter()
        with pytest.raises(AceError, match=text):
            nl.build(bad, cell, [1, 1, 1], 5.0)
        assert time.perf_counter() - t < 2.0
    # the list still works
    x = torch.tensor([[1.0, 2.0], [1.0, 1.0], [1.0, 1.0]], dtype=torch.float64, device="cuda:0")
    assert nl.build(x, cell, [1, 1, 1], 5.0).nnbr == 2
