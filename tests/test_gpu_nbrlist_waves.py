"""The wave-per-atom neighbour search on the GPU against the brute-force oracle
where its stretches can go wrong: more neighbours than a ring holds, counts
around 64, many images of one bin, rows cut by the cell's faces, atom counts
around a scan block of 2,048, an open axis beside periodic ones.  Whole
numbers are compared exactly; positions are sums of a few numbers below 100
(1e-12)."""
import numpy as np
import pytest
import torch

import nbr_oracle as N
from acehip.atoms import NeighbourList

pytestmark = pytest.mark.gpu

CASES = {
    "ring_wraps": (6.0 * np.eye(3), [1, 1, 1], 90, 4.6),         # about 170 neighbours, one or two bins per axis
    "about_64": (9.0 * np.eye(3), [1, 1, 1], 120, 4.5),
    "one_bin_many_images": (np.diag([1.1, 1.3, 1.2]), [1, 1, 1], 1, 5.0),
    "long_rows": (np.diag([40.0, 6.0, 6.0]), [1, 1, 1], 700, 2.9),
    "scan_block": (30.0 * np.eye(3), [1, 1, 1], 2048, 3.1),
    "scan_block_plus_1": (30.0 * np.eye(3), [1, 0, 1], 2049, 3.1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_wave_search(cuda, name):
    cell, pbc, n, rcut = CASES[name]
    print(f"[gpu] wave search {name}: {n} atoms, rcut {rcut}", flush=True)
    x = N.random_system(n, cell, pbc, seed=n)
    z = (np.arange(n) % 3).astype(np.int8)
    nl = NeighbourList(0).build(x, cell, pbc, rcut, z)
    i0, j0, S0, r0 = N.neighbour_pairs(x, cell, pbc, rcut)
    off, j, S, r = (t.cpu().numpy() for t in (nl.offsets, nl.nbr_j, nl.shift.T, nl.xyz.T))
    assert np.array_equal(off, N.offsets_of(i0, n))
    i = np.repeat(np.arange(n), np.diff(off))
    order = np.lexsort((S[:, 2], S[:, 1], S[:, 0], j, i))
    assert np.array_equal(j[order], j0) and np.array_equal(S[order], S0)
    assert np.max(np.abs(r[order] - r0)) < 1e-12
    assert np.array_equal(nl.species.cpu().numpy(), z[j])
    rev = nl.rev.cpu().numpy()
    assert np.array_equal(rev[rev], np.arange(len(rev)))
    assert np.array_equal(j[rev], i) and np.array_equal(S[rev], -S) and np.array_equal(r[rev], -r)
    # positions one step later, same pairs
    x1 = x + 0.05 * np.random.default_rng(1).normal(size=x.shape)
    nl.update(x1)
    assert np.max(np.abs(nl.xyz.cpu().numpy().T - (x1[j] - x1[i] + S @ cell))) < 1e-12
