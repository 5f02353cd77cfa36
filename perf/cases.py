"""Performance cases: the calls that programs built on this package make.

A case is a dict of plain values; ``listed()`` names the standing ones,
``draw(rng)`` gives more of the same ranges.  ``prepare`` makes the inputs on
the GPU, ``run`` is one pass through the public entry points, ``exact`` the
same outputs in 64 bits by plain torch, from the basis tables alone.

Kinds of case:

* ``sites``   energies, or energies and forces, of a batch of environments
              (:meth:`HIPEvaluator.energy`, :meth:`HIPEvaluator.energy_forces`);
* ``md``      one step of molecular dynamics on a periodic crystal: new
              positions in, energy, forces and virial out, through
              :class:`ACECalculator` (small cells) or through the device
              buffers of :class:`NeighbourList` (large ones);
* ``list``    building the neighbour list of a configuration;
* ``rows``    the energy and force rows of a least-squares fit
              (:meth:`ACECalculator.basis_energy_forces`);
* ``train``   gradient of an energy-and-force loss with respect to the
              coefficients (:func:`site_energies`, double backward);
* ``network`` values and input gradients of the learned surrogate's network
              (:meth:`MLPEnsemble.predict_grad`).
"""
from __future__ import annotations

import functools
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "ace.jl_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "ace.jl_amd"))

# The models, as the package's workloads define them (acehip/synth.py).
MODELS = {
    "o3d6": dict(order=3, maxdeg=6, L=4, prop="Invariant"),                       # 97 functions, 29 pooled values
    "o4d12": dict(order=4, maxdeg=12, L=6, prop="Invariant"),                     # 3235 functions, 139 pooled values
    "o4d14w": dict(order=4, maxdeg=14, L=10, prop="Invariant",
                   weight={"n": 1.0, "l": 1.5}),                                  # 2566 functions, 104 pooled values
    "o5d10": dict(order=5, maxdeg=10, L=4, prop="Invariant"),                     # 2664 functions, 84 pooled values
    "o3d10v2": dict(order=3, maxdeg=10, L=5, prop="EuclideanVector", species=2),  # 5408 functions, 220 pooled values
}
RCUT = 5.0
A_FCC = 3.6


def listed():
    return [
        # one environment at a time: a Monte Carlo move, or an atomistic code that calls per site
        dict(name="one_site", kind="sites", model="o3d6", nenv=1, nbrs=12, forces=True, waves=8, check=True),
        # a small periodic cell, one MD step through the calculator with its skin
        dict(name="md_cell", kind="md", model="o4d12", cells=4, skin=0.5, device=False),
        # a crystal of 55,296 atoms, one MD step on device buffers
        dict(name="md_crystal", kind="md", model="o4d12", cells=24, skin=0.0, device=True),
        # the benchmark's batch: 100,000 environments of about 30 neighbours, buffers checked once
        dict(name="sites_o4", kind="sites", model="o4d12", nenv=100000, nbrs=30, forces=True, waves=16, check=False),
        # energies alone, for the acceptance of moves or a data set's labels; every call checks its buffers
        dict(name="energies_o4", kind="sites", model="o4d12", nenv=20011, nbrs=30, forces=False, waves=16, check=True),
        # the reference's profiled model, 10 neighbours, high angular momenta
        dict(name="sites_weighted", kind="sites", model="o4d14w", nenv=50000, nbrs=10, forces=True, waves=16,
             check=True),
        # correlation order 5
        dict(name="sites_o5", kind="sites", model="o5d10", nenv=30011, nbrs=30, forces=True, waves=16, check=False),
        # two species, vector-valued: dipoles or forces as an equivariant property, with their Jacobians
        dict(name="sites_vector", kind="sites", model="o3d10v2", nenv=16385, nbrs=40, forces=True, waves=16,
             check=True),
        # the list build an MD run repeats when atoms have left the skin (the reach lies
        # between two shells, so that every seed has the same number of pairs)
        dict(name="list_build", kind="list", cells=24, reach=5.45, species=0),
        # energy and force rows of a fit, one cell
        dict(name="fit_rows", kind="rows", model="o4d12", cells=3),
        # gradient of an energy-and-force loss over a mini-batch
        dict(name="train_forces", kind="train", model="o4d12", nenv=2003, nbrs=30, waves=16, check=True),
        # the surrogate's network over a batch: 4 members, values and input gradients
        dict(name="network", kind="network", nenv=20011, members=4, inputs=151),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sites"] * 5 + ["md", "md", "list", "rows", "train", "network"])
    if kind == "sites":
        model = rng.choice(["o3d6", "o4d12", "o4d12", "o4d14w", "o5d10", "o3d10v2"])
        top = {"o3d6": 100000, "o4d12": 100000, "o4d14w": 60000, "o5d10": 50000, "o3d10v2": 20000}[model]
        return dict(kind=kind, model=model, nenv=_log(rng, 1, top), nbrs=rng.randint(8, 45),
                    forces=rng.random() < 0.75, waves=rng.choice([8, 16]), check=rng.random() < 0.5)
    if kind == "md":
        device = rng.random() < 0.5
        return dict(kind=kind, model=rng.choice(["o3d6", "o4d12", "o4d14w"]), cells=rng.randint(12, 24) if device
                    else rng.randint(4, 11), skin=0.0 if device else rng.choice([0.3, 0.5, 0.8]), device=device)
    if kind == "list":
        return dict(kind=kind, cells=rng.randint(3, 24), reach=rng.choice([4.75, 5.4, 5.95]),
                    species=rng.choice([0, 2]))
    if kind == "rows":
        return dict(kind=kind, model=rng.choice(["o3d6", "o4d14w"]), cells=rng.choice([3, 4]))
    if kind == "network":
        return dict(kind=kind, nenv=_log(rng, 64, 20000), members=rng.randint(1, 4), inputs=rng.randint(20, 160))
    return dict(kind=kind, model=rng.choice(["o3d6", "o4d12", "o4d14w"]), nenv=_log(rng, 50, 2000),
                nbrs=rng.randint(10, 45), waves=rng.choice([8, 16]), check=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs


@functools.lru_cache(maxsize=None)
def _basis(model):
    from acehip import synth
    basis = synth.make_basis(MODELS[model])
    return basis, synth.coefficients(len(basis), 17)


@functools.lru_cache(maxsize=None)
def _evaluator(model, waves, check):
    """One model is loaded once and evaluates many batches."""
    from acehip.evaluator import HIPEvaluator
    basis, c = _basis(model)
    ev = HIPEvaluator(basis, c, device=0, waves=waves)
    ev.set_validation(check)
    return ev


def _envs(case, seed):
    """Offsets, neighbour vectors (3, nnbr) and species of a batch: neighbour
    counts Poisson clipped to [5, 80] (in an order of the seed's, the same
    counts for every seed), isotropic directions, radii uniform in [0.8, 5.0],
    species equally likely."""
    n = case["nenv"]
    lens = np.clip(np.random.default_rng(case["nbrs"]).poisson(case["nbrs"], size=n), 5, 80)
    lens = np.random.default_rng(int(seed) + 3).permutation(lens)
    off = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), device="cuda")
    m = int(lens.sum())
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 11)
    d = torch.randn((3, m), dtype=torch.float64, device="cuda", generator=g)
    r = 0.8 + 4.2 * torch.rand(m, dtype=torch.float64, device="cuda", generator=g)
    xyz = d / d.square().sum(0).sqrt() * r
    nsp = MODELS[case["model"]].get("species", 0)
    sp = torch.randint(0, nsp, (m,), device="cuda", generator=g).to(torch.int8) if nsp else None
    return off, xyz, sp


def _crystal(cells, seed, sigma=0.1, flat=False):
    """FCC crystal of cells^3 conventional cells with Gaussian displacements,
    or flat ones (|d| <= sigma along each axis)."""
    base = 0.5 * A_FCC * np.array([[0, 0, 0], [0, 1, 1], [1, 0, 1], [1, 1, 0]], dtype=np.float64)
    k = np.arange(cells)
    g = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    x = (g[:, None, :] * A_FCC + base[None]).reshape(-1, 3)
    rng = np.random.default_rng(int(seed) + 101)
    x = x + sigma * (rng.uniform(-1, 1, size=x.shape) if flat else rng.standard_normal(x.shape))
    return x, np.diag(np.full(3, cells * A_FCC))


def _step(x, seed, size=0.02):
    """Positions one MD step later."""
    return x + size * np.clip(np.random.default_rng(int(seed) + 977).standard_normal(x.shape), -3, 3)


def _net(case):
    """Weights of the ensemble, one list of (W, b) per member, and their flat
    FP32 layout W1[128][160], b1, W2[128][128], b2, W3[128][128], b3, w4[128], b4."""
    rng = np.random.default_rng(23)
    nets, flat = [], []
    for _ in range(case["members"]):
        net = []
        for rows, cols, used in ((128, 160, case["inputs"]), (128, 128, 128), (128, 128, 128), (1, 128, 128)):
            W = np.zeros((rows, cols), dtype=np.float32)
            W[:, :used] = rng.uniform(-1, 1, size=(rows, used)) * np.sqrt(6.0 / used)
            net.append((W, rng.uniform(-0.1, 0.1, size=rows).astype(np.float32)))
        nets.append(net)
        p = np.concatenate([v.reshape(-1) for layer in net for v in layer])
        flat.append(np.concatenate([p, np.zeros(-len(p) % 16, dtype=np.float32)]))
    return nets, np.concatenate(flat)


def _net_inputs(case, seed):
    """Normalised features in BF16, zero past the inputs."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 13 + 3)
    X = torch.zeros((case["nenv"], 160), dtype=torch.bfloat16, device="cuda")
    X[:, :case["inputs"]] = torch.randn((case["nenv"], case["inputs"]), device="cuda", generator=g).to(torch.bfloat16)
    return X


def _targets(case, seed, xyz):
    """Energies and gradients that a loss compares with."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 31 + 5)
    return (0.1 * torch.randn(case["nenv"], dtype=torch.float64, device="cuda", generator=g),
            0.1 * torch.randn(xyz.shape, dtype=torch.float64, device="cuda", generator=g))


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "network":
        from acehip.mlp import MLPEnsemble
        net = MLPEnsemble(nmemb=case["members"], nin=case["inputs"])
        net.set_params(_net(case)[1])
        s.update(net=net, X=_net_inputs(case, seed))
        return s
    if kind in ("sites", "train"):
        from acehip.evaluator import EnvBatch
        ev = _evaluator(case["model"], case["waves"], case["check"])
        off, xyz, sp = _envs(case, seed)
        s.update(ev=ev, batch=EnvBatch(off, xyz, sp))
        if kind == "sites":
            nc = 1 if ev.prop == 0 else 3
            s["E"] = torch.empty((case["nenv"],) if nc == 1 else (case["nenv"], 3), dtype=torch.float64, device="cuda")
            s["dE"] = torch.empty((3 * nc, xyz.shape[1]), dtype=torch.float64, device="cuda") if case["forces"] else None
        if kind == "train":
            s["E0"], s["F0"] = _targets(case, seed, xyz)
            s["c"] = torch.as_tensor(_basis(case["model"])[1], device="cuda")
        return s
    from acehip.atoms import ACECalculator, Atoms, NeighbourList
    x, cell = _crystal(case["cells"], seed, *((0.05, True) if kind == "list" else ()))
    if kind == "list":
        s.update(nl=NeighbourList(0), cell=cell, pos=torch.as_tensor(x.T.copy(), device="cuda"))
        if case["species"]:
            z = np.random.default_rng(int(seed) + 5).integers(0, case["species"], size=len(x)).astype(np.int8)
            s["z"] = torch.as_tensor(z, device="cuda")
        return s
    if kind == "rows":
        s.update(calc=ACECalculator(_evaluator(case["model"], 16, True), rcut=RCUT), at=Atoms(x, cell))
        return s
    # md: the list of the last build, and the positions of the next step
    x1 = _step(x, seed)
    if case["device"]:
        ev = _evaluator(case["model"], 16, False)
        nl = NeighbourList(0)
        nl.build(torch.as_tensor(x.T.copy(), device="cuda"), cell, (1, 1, 1), RCUT)
        s.update(ev=ev, nl=nl, batch=nl.batch(), pos=torch.as_tensor(x1.T.copy(), device="cuda"),
                 E=torch.empty(nl.natoms, dtype=torch.float64, device="cuda"),
                 dE=torch.empty((3, nl.nnbr), dtype=torch.float64, device="cuda"),
                 F=torch.empty((3, nl.natoms), dtype=torch.float64, device="cuda"))
    else:
        calc = ACECalculator(_evaluator(case["model"], 8, True), rcut=RCUT, skin=case["skin"])
        calc.energy(Atoms(x, cell))  # the list is there when the step begins
        s.update(calc=calc, at=Atoms(x1, cell))
    return s


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "sites":
        if case["forces"]:
            return s["ev"].energy_forces(s["batch"], s["E"], s["dE"])
        return s["ev"].energy(s["batch"], s["E"])
    if kind == "md":
        if case["device"]:
            s["nl"].update(s["pos"])
            s["ev"].energy_forces(s["batch"], s["E"], s["dE"])
            F, W = s["nl"].forces(s["dE"], s["F"], virial=True)
            return dict(E=s["E"], F=F, W=W)
        E, F, W = s["calc"].energy_forces(s["at"], virial=True)
        return dict(E=E, F=F, W=W)
    if kind == "list":
        nl = s["nl"].build(s["pos"], s["cell"], (1, 1, 1), case["reach"], s.get("z"))
        out = dict(offsets=nl.offsets, nbr_j=nl.nbr_j, shift=nl.shift, xyz=nl.xyz, rev=nl.rev)
        if nl.species is not None:
            out["species"] = nl.species
        return out
    if kind == "network":
        return s["net"].predict_grad(s["X"])
    if kind == "rows":
        EB, FB = s["calc"].basis_energy_forces(s["at"])
        return dict(EB=EB, FB=FB)
    # train: loss = sum (E - E0)^2 + sum |dE/dr - F0|^2
    from acehip.autograd import site_energies
    b = s["batch"]
    c = s["c"].clone().requires_grad_(True)
    x = b.xyz.clone().requires_grad_(True)
    E = site_energies(s["ev"], c, b.offsets, x, b.species)
    (dE,) = torch.autograd.grad(E.sum(), x, create_graph=True)
    loss = (E - s["E0"]).square().sum() + (dE - s["F0"]).square().sum()
    (gc,) = torch.autograd.grad(loss, c)
    return dict(E=E.detach(), dE=dE.detach(), grad_c=gc)


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _sizes(model):
    basis, _ = _basis(model)
    from acehip.tables import basis_tables
    T = basis_tables(basis)
    npool = len({(int(a[0]), int(a[1]), int(a[2]), abs(int(a[3]))) for a in T["aspec"]})
    return dict(nAA=len(T["orders"]), nB=int(T["a2b"]["shape"][0]), nnz=len(T["a2b"]["vals"]), npool=npool,
                nr=len(T["rn"]["A"]), np=(T["L"] + 1) * (T["L"] + 2) // 2, vec=T["prop"] != "Invariant")


def _fcc_neighbours(rcut):
    k = np.arange(-4, 5)
    base = 0.5 * A_FCC * np.array([[0, 0, 0], [0, 1, 1], [1, 0, 1], [1, 1, 0]], dtype=np.float64)
    g = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3) * A_FCC
    r = np.linalg.norm((g[:, None] + base[None]).reshape(-1, 3), axis=1)
    return int(((r > 0) & (r < rcut)).sum())


def work(case):
    """Inputs read once, outputs written once.  Per neighbour the radial and
    angular values and their sum into the pooled values (twice that with
    gradients); per AA function one multiply-add on a product that its mirror
    image shares (2 flops), three times that with the adjoint, the component
    count times that for a vector property."""
    kind = case["kind"]
    if kind == "list":
        n = 4 * case["cells"] ** 3
        m = n * _fcc_neighbours(case["reach"])
        return {"bytes": 24.0 * n + m * (4 + 12 + 24 + 4), "flops": 10.0 * m}
    if kind == "network":
        n, k = case["nenv"], case["members"]
        w = 128.0 * (case["inputs"] + 128 + 128 + 1)
        return {"bytes": n * (2.0 * 160 + k * 4 + k * 4 * 160) + 4 * k * w, "flops": n * k * 4 * w}
    z = _sizes(case["model"])
    vec = 3 if z["vec"] else 1
    if kind in ("md", "rows"):
        n = 4 * case["cells"] ** 3
        m = n * _fcc_neighbours(RCUT)
    else:
        n, m = case["nenv"], case["nenv"] * max(5, case["nbrs"])
    one = 5 * z["nr"] + 8 * z["np"] + 10 + 4 * z["npool"]
    e_flops, f_flops = m * one + 2.0 * vec * n * z["nAA"], 2 * m * one + 4.0 * vec * n * z["nAA"]
    base = 24.0 * m + 4.0 * n
    if kind == "sites":
        out = 8.0 * vec * n + (24.0 * vec * m if case["forces"] else 0.0)
        return {"bytes": base + out, "flops": e_flops + (f_flops if case["forces"] else 0.0)}
    if kind == "md":
        return {"bytes": 24.0 * n + 16.0 * m + 32.0 * n, "flops": e_flops + f_flops}
    if kind == "rows":
        return {"bytes": 24.0 * n + 8.0 * z["nB"] * (1 + 3.0 * n), "flops": 3 * m * one + 8.0 * m * z["nB"] * 3}
    return {"bytes": 2 * base + 24.0 * m + 8.0 * z["nB"], "flops": 2 * (e_flops + f_flops)}


# ---------------------------------------------------------------------------
# the same in 64 bits, from the basis tables


class _Plain:
    """A = sum_j R_n Y_lm, AA = prod A, B = A2B AA, E = c . B in plain torch."""

    def __init__(self, model):
        from acehip.tables import basis_tables
        basis, c = _basis(model)
        T = basis_tables(basis)
        dev = "cuda"
        self.rn, self.L = T["rn"], T["L"]
        self.aspec = torch.as_tensor(np.asarray(T["aspec"]), device=dev)
        self.nA = len(self.aspec)
        o = np.asarray(T["orders"])
        idx = np.asarray(T["iAA2iA"]).astype(np.int64).copy()
        for q in range(idx.shape[1]):
            idx[q >= o, q] = self.nA  # the constant 1
        self.orders, self.idx = o, torch.as_tensor(idx, device=dev)
        self.nB, self.nAA = (int(v) for v in T["a2b"]["shape"])
        rows, cols = np.asarray(T["a2b"]["rows"]), np.asarray(T["a2b"]["cols"])
        vals = np.asarray(T["a2b"]["vals"])
        self.vec = T["prop"] != "Invariant"
        vals = vals.reshape(len(rows), -1).astype(np.complex128)
        self.nc = vals.shape[1]
        ct = np.zeros((self.nAA, self.nc), dtype=np.complex128)
        np.add.at(ct, cols, vals * c[rows][:, None])
        self.ct = torch.as_tensor(ct, device=dev)
        order = np.lexsort((cols, rows))
        self.rows = torch.as_tensor(rows[order], device=dev)
        self.cols = torch.as_tensor(cols[order], device=dev)
        self.vals = torch.as_tensor(vals[order], device=dev)

    def phi(self, x, sp, dx=None):
        """1p values [nnbr, nA] of neighbour vectors x [nnbr, 3], with dx also
        their derivative along dx (every quantity with its differential)."""
        d = dx is not None
        dx = dx if d else torch.zeros_like(x)
        rn = self.rn
        r = x.square().sum(1).sqrt()
        dr = (x * dx).sum(1) / r
        t = ((1.0 + rn["r0"]) / (1.0 + r)) ** rn["p"]
        dt = -rn["p"] * t / (1.0 + r) * dr
        pl, pr = int(rn["pl"]), int(rn["pr"])
        a, b = t - rn["tl"], t - rn["tr"]
        cut = a ** pl * b ** pr
        dcut = ((pl * a ** (pl - 1) * b ** pr if pl else 0.0) + (pr * a ** pl * b ** (pr - 1) if pr else 0.0)) * dt
        out = torch.zeros_like(t, dtype=torch.bool)
        if pl > 0:
            out |= a < 0
        if pr > 0:
            out |= b > 0
        cut, dcut = cut.masked_fill(out, 0.0), dcut.masked_fill(out, 0.0)
        A, B, C = rn["A"], rn["B"], rn["C"]
        R, dR = [float(A[0]) * cut], [float(A[0]) * dcut]
        for n in range(1, len(A)):
            al = float(A[n]) * t + float(B[n])
            v, dv = al * R[-1], al * dR[-1] + float(A[n]) * dt * R[-1]
            if n > 1:
                v, dv = v + float(C[n]) * R[-2], dv + float(C[n]) * dR[-2]
            R.append(v)
            dR.append(dv)
        # Y_lm = Q_lm(cos theta) ((x + i y) / r)^m, Q_lm = P_lm / sin^m
        ct = x[:, 2] / r
        dct = (dx[:, 2] - ct * dr) / r
        e = torch.complex(x[:, 0], x[:, 1]) / r
        de = (torch.complex(dx[:, 0], dx[:, 1]) - e * dr) / r
        Y, dY = {}, {}
        Qmm = float(np.sqrt(0.25 / np.pi))
        em, dem = torch.ones_like(e), torch.zeros_like(e)
        for m in range(self.L + 1):
            if m:
                Qmm = -float(np.sqrt(1.0 + 0.5 / m)) * Qmm
                em, dem = em * e, dem * e + em * de
            Qa, Qb = torch.zeros_like(r), torch.full_like(r, Qmm)
            dQa, dQb = torch.zeros_like(r), torch.zeros_like(r)
            for l in range(m, self.L + 1):
                if l > m:
                    k = float(np.sqrt((4.0 * l * l - 1) / (l * l - m * m)))
                    h = float(np.sqrt(((l - 1.0) ** 2 - m * m) / (4 * (l - 1.0) ** 2 - 1))) if l > m + 1 else 0.0
                    Qa, Qb, dQa, dQb = Qb, k * (ct * Qb - h * Qa), dQb, k * (dct * Qb + ct * dQb - h * dQa)
                Y[l, m], dY[l, m] = Qb * em, dQb * em + Qb * dem
                if m:
                    Y[l, -m] = ((-1) ** m * Y[l, m].conj()).resolve_conj()
                    dY[l, -m] = ((-1) ** m * dY[l, m].conj()).resolve_conj()
        spec = [(int(v[1]) - 1, (int(v[2]), int(v[3]))) for v in self.aspec.cpu().numpy()]
        mu = self.aspec[:, 0]
        keep = sp[:, None].long() == mu[None, :] if sp is not None and int(mu.max()) >= 0 else None
        v = torch.stack([Y[lm] * R[n] for n, lm in spec], 1)
        dv = torch.stack([dY[lm] * R[n] + Y[lm] * dR[n] for n, lm in spec], 1) if d else None
        if keep is not None:
            v = v.masked_fill(~keep, 0.0)
            dv = dv.masked_fill(~keep, 0.0) if d else None
        return (v, dv) if d else v

    def pooled(self, phi, own, n):
        """A [nA, n] of the environments ``own`` assigns the neighbours to."""
        A = torch.zeros((n, 2 * self.nA), dtype=torch.float64, device=phi.device)
        A.index_add_(0, own, torch.view_as_real(phi).reshape(len(own), -1))
        return torch.view_as_complex(A.view(n, self.nA, 2)).t().contiguous()

    @staticmethod
    def _with(A, value):
        return torch.cat([A, torch.full((1, A.shape[1]), value, dtype=A.dtype, device=A.device)])

    def products(self, A, dA=None):
        """AA [nAA, n], with dA also its directional derivative."""
        A1 = self._with(A, 1.0)
        p = A1[self.idx[:, 0]]
        if dA is None:
            for q in range(1, self.idx.shape[1]):
                p = p * A1[self.idx[:, q]]
            return p
        d1 = self._with(dA, 0.0)
        dp = d1[self.idx[:, 0]]
        for q in range(1, self.idx.shape[1]):
            a, da = A1[self.idx[:, q]], d1[self.idx[:, q]]
            dp, p = dp * a + p * da, p * a
        return p, dp

    def energies(self, A, adjoint):
        """E [nc, n], and with ``adjoint`` G [nc, nA, n], dE_p = Re sum G dA."""
        p = self.products(A)
        E = (self.ct.t() @ p).real
        if not adjoint:
            return E, None
        A1, n = self._with(A, 1.0), A.shape[1]
        G = torch.zeros((self.nc, self.nA + 1, 2 * n), dtype=torch.float64, device=A.device)
        for q in range(self.idx.shape[1]):
            w = None
            for t in range(self.idx.shape[1]):
                if t != q:
                    f = A1[self.idx[:, t]]
                    w = f if w is None else w * f
            for k in range(self.nc):
                G[k].index_add_(0, self.idx[:, q], torch.view_as_real(w * self.ct[:, k, None]).reshape(self.nAA, -1))
        return E, torch.view_as_complex(G.view(self.nc, self.nA + 1, n, 2))[:, :self.nA]

    def values(self, p):
        """Re A2B p [nB, n] of products p [nAA, n]."""
        out = torch.zeros((self.nB, p.shape[1]), dtype=torch.float64, device=p.device)
        return out.index_add_(0, self.rows, (self.vals[:, :1] * p[self.cols]).real)

    def gradients(self, x, sp):
        """dphi / dx_d [3, nnbr, nA]."""
        out = []
        for d in range(3):
            t = torch.zeros_like(x)
            t[:, d] = 1.0
            out.append(self.phi(x, sp, t)[1])
        return torch.stack(out)


@functools.lru_cache(maxsize=1)
def _plain(model):
    return _Plain(model)


def _chunks(off, nAA, budget=2.5e8):
    n = len(off) - 1
    step = max(1, int(budget / (16.0 * nAA)) * 4)
    for a in range(0, n, step):
        b = min(n, a + step)
        yield a, b, int(off[a]), int(off[b])


def _exact_sites(P, off, xyz, sp, forces):
    oh = off.cpu().numpy()
    Es, Gs = [], []
    x = xyz.t()
    for a, b, j0, j1 in _chunks(oh, P.nAA):
        own = torch.repeat_interleave(torch.arange(b - a, device="cuda"), (off[a + 1:b + 1] - off[a:b]).long())
        xc, sc = x[j0:j1].contiguous(), None if sp is None else sp[j0:j1]
        phi = P.phi(xc, sc)
        E, G = P.energies(P.pooled(phi, own, b - a), forces)
        Es.append(E.t())
        if forces:
            d = P.gradients(xc, sc)
            Gs.append(torch.stack([(G[k].t()[own] * d[q]).sum(1).real for k in range(P.nc) for q in range(3)]))
    E = torch.cat(Es)
    return (E if P.vec else E[:, 0].contiguous()), torch.cat(Gs, 1) if forces else None


def _pairs(x, box, rcut):
    """Environments of a cubic periodic cell (edge at least 2 rcut):
    offsets, neighbour index, vectors (3, nnbr)."""
    n = len(x)
    off, J, V = [0], [], []
    step = max(1, int(4e7 // n))
    for a in range(0, n, step):
        d = x[None, :, :] - x[a:a + step, None, :]
        d = d - box * torch.round(d / box)
        r2 = d.square().sum(2)
        i, j = torch.nonzero((r2 < rcut * rcut) & (r2 > 0), as_tuple=True)
        V.append(d[i, j])
        J.append(j)
        off.append(torch.bincount(i, minlength=min(step, n - a)))
    lens = torch.cat(off[1:])
    o = torch.zeros(n + 1, dtype=torch.long, device=x.device)
    o[1:] = torch.cumsum(lens, 0)
    return o, torch.cat(J), torch.cat(V).t().contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "list":
        return None  # the order of a list's entries is the builder's own
    if kind == "network":
        X = _net_inputs(case, seed).double()
        ys, gs = [], []
        for net in _net(case)[0]:
            x = X.clone().requires_grad_(True)
            h = x
            for i, (W, b) in enumerate(net):
                h = h @ torch.as_tensor(W, device="cuda").double().t() + torch.as_tensor(b, device="cuda").double()
                if i < 3:
                    h = h * torch.sigmoid(h)
            (g,) = torch.autograd.grad(h.sum(), x)
            ys.append(h.detach()[:, 0])
            gs.append(g)
        return torch.stack(ys), torch.stack(gs)
    P = _plain(case["model"])
    if kind in ("sites", "train"):
        off, xyz, sp = _envs(case, seed)
        if kind == "sites":
            E, dE = _exact_sites(P, off, xyz, sp, case["forces"])
            return (E, dE) if case["forces"] else E
        oh = off.cpu().numpy()
        x = xyz.t()
        E0, F0 = _targets(case, seed, xyz)
        E, dE = _exact_sites(P, off, xyz, sp, True)
        wE, wF = 2 * (E - E0), 2 * (dE - F0).t().contiguous()
        gc = torch.zeros(P.nB, dtype=torch.float64, device="cuda")
        for a, b, j0, j1 in _chunks(oh, P.nAA):
            own = torch.repeat_interleave(torch.arange(b - a, device="cuda"), (off[a + 1:b + 1] - off[a:b]).long())
            xc = x[j0:j1].contiguous()
            phi, dphi = P.phi(xc, None, wF[j0:j1])
            p, dp = P.products(P.pooled(phi, own, b - a), P.pooled(dphi, own, b - a))
            gc += P.values((p * wE[a:b] + dp).sum(1, keepdim=True))[:, 0]
        return dict(E=E, dE=dE, grad_c=gc)
    x, cell = _crystal(case["cells"], seed)
    box = float(cell[0, 0])
    if box < 2 * RCUT:
        return None
    if kind == "md":
        # the pairs of the list: those of the build for device buffers, those
        # within the cutoff (others contribute nothing) with a skin
        x1 = torch.as_tensor(_step(x, seed), device="cuda")
        off, J, V = _pairs(torch.as_tensor(x, device="cuda"), box, RCUT + case["skin"])
        own = torch.repeat_interleave(torch.arange(len(x1), device="cuda"), off[1:] - off[:-1])
        d = x1[J] - x1[own]
        V = (d + box * torch.round((V.t() - d) / box)).t().contiguous()
        E, g = _exact_sites(P, off, V, None, True)
        F = torch.zeros((len(x1), 3), dtype=torch.float64, device="cuda")
        F.index_add_(0, own, g.t()).index_add_(0, J, -g.t())
        W = -(g @ V.t())
        if case["device"]:
            return dict(E=E, F=F.t().contiguous(), W=W)
        return dict(E=float(E.sum()), F=F.cpu().numpy(), W=W.cpu().numpy())
    # rows: the summed basis and its gradients with respect to the atoms
    xt = torch.as_tensor(x, device="cuda")
    off, J, V = _pairs(xt, box, RCUT)
    n = len(xt)
    EB = torch.zeros(P.nB, dtype=torch.float64, device="cuda")
    FB = torch.zeros((n, P.nB, 3), dtype=torch.float64, device="cuda")
    for i in range(n):
        j0, j1 = int(off[i]), int(off[i + 1])
        xc = V[:, j0:j1].t().contiguous()
        A = P.phi(xc, None).sum(0)[:, None].contiguous()
        EB += P.values(P.products(A))[:, 0]
        A1 = P._with(A, 1.0)[:, 0]
        D = torch.zeros((P.nAA, P.nA + 1), dtype=torch.complex128, device="cuda")  # dAA / dA
        at = torch.arange(P.nAA, device="cuda")
        for q in range(P.idx.shape[1]):
            w = torch.ones(P.nAA, dtype=torch.complex128, device="cuda")
            for t in range(P.idx.shape[1]):
                if t != q:
                    w = w * A1[P.idx[:, t]]
            D[at, P.idx[:, q]] += w
        M = torch.zeros((P.nB, 2 * P.nA), dtype=torch.float64, device="cuda")
        M.index_add_(0, P.rows, torch.view_as_real(P.vals * D[P.cols, :P.nA]).reshape(len(P.rows), -1))
        M = torch.view_as_complex(M.view(P.nB, P.nA, 2))
        g = torch.stack([(M @ d.t()).real for d in P.gradients(xc, None)], 2)  # [nB, nnbr, 3]
        FB[i] += g.sum(1)
        FB.index_add_(0, J[j0:j1], -g.permute(1, 0, 2).contiguous())
    return dict(EB=EB, FB=FB.permute(1, 0, 2).contiguous())
