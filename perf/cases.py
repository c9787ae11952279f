"""Performance cases of the Behler-Parrinello path: what a program that uses this
package has it do, at the sizes of the package's own workloads.

A case is a dict of plain values; ``kind`` names the call sequence:

  ef        neighbour build + energies, forces and virials of a batch of
            periodic structures (single-point evaluation, active learning,
            minimisation): ``Engine.neighbors`` + ``Engine.energy_forces``;
  energies  neighbour build + energies only (validation error of a training
            set): ``Engine.neighbors`` + ``Engine.energies``;
  train     one energy + force training step with Adam.  ``resident`` > batch
            size: every step draws its structures from a resident set (gather,
            set-up, list, step); otherwise the batch and its list are fixed
            (full-batch training on a small set);
  md        a velocity-Verlet segment from a given start: list at rc + skin,
            then ``steps`` steps on it;
  pair      the LAMMPS-style interface on host arrays: one call with a new
            list, then calls that reuse it while the atoms move.

``prepare`` makes structures, potentials and labels from the seed with numpy and
torch alone; ``exact`` evaluates the same definitions in FP64 with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

# ------------------------------------------------------------------ cases


def listed():
    return [
        # one 64-molecule water box: the smallest call, bound by latency (one
        # structure per call: relaxations, dimers, interactive use)
        {"name": "ef_water_1x192", "kind": "ef", "basis": "water", "structures": 1, "molecules": 64, "uneven": False,
         "scaled": False},
        # the ordinary evaluation batch: 64 water boxes of 192 atoms
        {"name": "ef_water_64x192", "kind": "ef", "basis": "water", "structures": 64, "molecules": 64, "uneven": False,
         "scaled": False},
        # a whole data set at once: 512 strained (triclinic) cells of 32 to 1024 atoms
        {"name": "ef_water_uneven_512", "kind": "ef", "basis": "water", "structures": 512, "molecules": 176,
         "uneven": True, "scaled": False},
        # a trained potential: inputs standardised over the set (bias -mean, scale
        # 1/deviation), which takes the inputs in FP64
        {"name": "ef_water_scaled_32x192", "kind": "ef", "basis": "water", "structures": 32, "molecules": 64,
         "uneven": False, "scaled": True},
        # argon, angular exponents up to 5 (the moment form's largest), 16 boxes of 256 atoms
        {"name": "ef_ar_zeta5_16x256", "kind": "ef", "basis": "ar5", "structures": 16, "cells": 4},
        # argon, angular exponents up to 8 (sums over triplets), 16 boxes of 256 atoms
        {"name": "ef_ar_zeta8_16x256", "kind": "ef", "basis": "ar8", "structures": 16, "cells": 4},
        # validation error of a training set: forward only, three species, 512 structures
        {"name": "energies_lips_512", "kind": "energies", "basis": "lips", "structures": 512},
        # the trainer's usual batch (32), drawn from a resident set on every step
        {"name": "train_lips_32_of_256", "kind": "train", "basis": "lips", "structures": 32, "resident": 256},
        # full-batch training on 128 structures with a fixed list
        {"name": "train_lips_128", "kind": "train", "basis": "lips", "structures": 128, "resident": 128},
        # a small MD cell: 2,048 atoms, one list and ten steps on it
        {"name": "md_water_2k", "kind": "md", "basis": "water", "reps": 2, "steps": 10},
        # large-scale MD: 1,048,576 atoms, one list and five steps on it
        {"name": "md_water_1m", "kind": "md", "basis": "water", "reps": 16, "steps": 5},
        # an MD host code: 1,536 owned atoms and their ghosts, a new list and nine steps on it
        {"name": "pair_water_1536", "kind": "pair", "basis": "water", "molecules": 512, "calls": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["water", "water", "scaled", "argon", "energies", "train", "train", "md", "md", "pair"])
    if kind == "water":
        total = _log_int(rng, 64, 40000)                    # molecules of the batch
        mol = min(total, _log_int(rng, 16, 341))
        s = max(1, total // mol)
        return {"kind": "ef", "basis": "water", "structures": s, "molecules": mol, "uneven": s >= 16 and rng.random() < 0.5,
                "scaled": False}
    if kind == "scaled":
        return {"kind": "ef", "basis": "water", "structures": _log_int(rng, 4, 96), "molecules": _log_int(rng, 32, 160),
                "uneven": False, "scaled": True}
    if kind == "argon":
        return {"kind": "ef", "basis": rng.choice(["ar5", "ar8"]), "structures": _log_int(rng, 1, 48),
                "cells": rng.randint(4, 6)}
    if kind == "energies":
        return {"kind": "energies", "basis": "lips", "structures": _log_int(rng, 16, 512)}
    if kind == "train":
        b = _log_int(rng, 8, 128)
        return {"kind": "train", "basis": "lips", "structures": b,
                "resident": b if rng.random() < 0.4 else min(256, b * rng.randint(2, 8))}
    if kind == "md":
        return {"kind": "md", "basis": "water", "reps": rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 10, 12]),
                "steps": rng.randint(5, 12)}
    return {"kind": "pair", "basis": "water", "molecules": _log_int(rng, 100, 1000), "calls": rng.randint(5, 12)}


# ------------------------------------------------------------------ potentials
# rs in Angstrom, radial width eta in 1/Angstrom (exp(-(eta (r - rs))^2)), angular
# width in Angstrom (exp(-(rij^2 + rik^2) / eta^2)); the same functions for every
# pair and triplet of species.  evac: energies of the isolated atoms in eV.

RC = 6.0


def _basis(name):
    if name == "water":
        rs = np.linspace(0.8, 6.0, 16)
        return {"species": ["H", "O"], "mass": [1.008, 15.999], "evac": [-13.6, -432.0], "cut": "TANH", "rs": rs,
                "reta": np.full(16, 1.0 / (rs[1] - rs[0])), "aeta": np.repeat([1.5, 2.5, 4.0, 6.0], 4),
                "zeta": np.tile([1.0, 1.0, 4.0, 4.0], 4), "lam": np.tile([1, -1], 8), "hidden": [32, 32],
                "neuron": "SOFTPLUS"}
    if name == "lips":
        rs = np.linspace(1.0, 6.0, 8)
        return {"species": ["Li", "P", "S"], "mass": [6.94, 30.97, 32.06], "evac": [-7.5, -178.0, -277.0],
                "cut": "TANH", "rs": rs, "reta": np.full(8, 1.0 / (rs[1] - rs[0])),
                "aeta": np.repeat([2.0, 3.5, 5.0], 4), "zeta": np.tile([1.0, 1.0, 2.0, 2.0], 3),
                "lam": np.tile([1, -1], 6), "hidden": [48, 48], "neuron": "TANH"}
    if name == "ar5":
        rs = np.linspace(1.0, 5.5, 10)
        return {"species": ["Ar"], "mass": [39.948], "evac": [-575.0], "cut": "COS", "rs": rs,
                "reta": np.full(10, 1.0 / (rs[1] - rs[0])), "aeta": np.repeat([1.5, 2.5, 4.0], 4),
                "zeta": np.tile([1.0, 2.0, 5.0, 5.0], 3), "lam": np.tile([1, -1, -1, 1], 3), "hidden": [24, 24],
                "neuron": "TANH"}
    if name == "ar8":
        return {"species": ["Ar"], "mass": [39.948], "evac": [-575.0], "cut": "COS",
                "rs": 1.0 + np.arange(8) * 5.0 / 7.0, "reta": np.full(8, math.sqrt(0.5)), "aeta": np.full(8, 10.0),
                "zeta": np.repeat([1.0, 2.0, 4.0, 8.0], 2), "lam": np.tile([1, -1], 4), "hidden": [20, 20],
                "neuron": "TANH"}
    raise ValueError(name)


def _potential(name, seed):
    """Basis and random networks: biases small, weights uniform with the Xavier spread."""
    pot = _basis(name)
    rng = np.random.default_rng([seed, 1])
    S = len(pot["species"])
    nin = S * len(pot["rs"]) + S * (S + 1) // 2 * len(pot["aeta"])
    pot["nin"], pot["layers"] = nin, []
    for _ in range(S):
        sizes, layers = [nin] + pot["hidden"] + [1], []
        for ni, no in zip(sizes[:-1], sizes[1:]):
            s = math.sqrt(2.0 / (ni + no))
            layers.append((rng.uniform(-math.sqrt(3.0) * s, math.sqrt(3.0) * s, size=(no, ni)), rng.normal(0.0, 0.001 * s, size=no)))
        pot["layers"].append(layers)
    pot["inpw"] = [np.ones(nin) for _ in range(S)]
    pot["inpb"] = [np.zeros(nin) for _ in range(S)]
    return pot


def _pack(layers):
    """One network's parameters: every bias, then every weight matrix column by column."""
    return np.concatenate([b for _, b in layers] + [w.T.reshape(-1) for w, _ in layers])


def _model(pot):
    from ann_amd.model import ANG, CUT, NEURON, RAD, Model, Network
    S = len(pot["species"])
    rad = (RAD["GAUSSIAN"], pot["rs"], pot["reta"])
    ang = (ANG["GAUSS"], pot["aeta"], pot["zeta"], pot["lam"])
    nets = [Network(nin=pot["nin"], nodes=pot["hidden"] + [1], neuron=NEURON[pot["neuron"]], c=1.0,
                    params=_pack(pot["layers"][a]), inpw=pot["inpw"][a], inpb=pot["inpb"][a]) for a in range(S)]
    return Model(pot["species"], np.array(pot["mass"]), np.array(pot["evac"]), RC, CUT[pot["cut"]],
                 [[rad] * S for _ in range(S)], [[ang] * (S * (S + 1) // 2) for _ in range(S)], nets)


# ------------------------------------------------------------------ structures
# a structure is (pos [n, 3], cell [3, 3] with the lattice vectors as columns, species [n])


def _molecules(rng, nmol, L, extra=0):
    """Water on a jittered grid, randomly turned, bonds near 0.96 A; ``extra`` single H."""
    ng = int(math.ceil(nmol ** (1.0 / 3.0) - 1e-9))
    while ng ** 3 < nmol + extra:
        ng += 1
    site = np.sort(rng.choice(ng ** 3, size=nmol + extra, replace=False))
    site = np.stack([site // (ng * ng), site // ng % ng, site % ng], 1)
    site = (site + 0.5) * (L / ng) + rng.normal(0.0, 0.1, size=(nmol + extra, 3))
    q = rng.normal(size=(nmol, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    ex = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w)], 1)
    ez = np.stack([2 * (x * z + y * w), 2 * (y * z - x * w), 1 - 2 * (x * x + y * y)], 1)
    th = math.radians(104.5) / 2
    bond = 0.96 + rng.normal(0.0, 0.02, size=(2, nmol, 1))
    h1 = bond[0] * (math.sin(th) * ex + math.cos(th) * ez)
    h2 = bond[1] * (-math.sin(th) * ex + math.cos(th) * ez)
    o = site[:nmol]
    pos = np.stack([o, o + h1, o + h2], 1).reshape(-1, 3)
    spc = np.tile(np.array([1, 0, 0], np.int32), nmol)
    return np.concatenate([pos, site[nmol:]]), np.concatenate([spc, np.zeros(extra, np.int32)])


def _water_batch(case, rng):
    out, sizes = [], np.random.default_rng([case["structures"], case["molecules"]])    # sizes belong to the case
    for _ in range(case["structures"]):
        if case["uneven"]:      # whole molecules, 32 to 6 * molecules - 32 atoms, 0.9 g/cm^3, strained
            nmol = max(1, int(round(sizes.integers(32, max(33, 6 * case["molecules"] - 32) + 1) / 3)))
            L = (nmol * 18.015 / 0.602214076 / 0.9) ** (1.0 / 3.0)
        else:
            nmol = case["molecules"]
            L = 12.42 * (nmol / 64.0) ** (1.0 / 3.0)
        pos, spc = _molecules(rng, nmol, L)
        strain = np.eye(3)
        if case["uneven"]:
            e = rng.uniform(-0.1, 0.1, size=(3, 3))
            strain = strain + 0.5 * (e + e.T)
        out.append((pos @ strain.T, strain * L, spc))
    return out


def _argon_batch(case, rng):
    c, a = case["cells"], 22.98 / 4
    fcc = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    g = np.stack(np.meshgrid(*[np.arange(c)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = ((g[:, None] + fcc) * a).reshape(-1, 3)
    return [(pos + rng.normal(0.0, 0.15, size=pos.shape), np.eye(3) * (c * a), np.zeros(len(pos), np.int32))
            for _ in range(case["structures"])]


def _lips_batch(n, rng):
    a = 5.6
    fcc = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    shapes = [(x, y, z) for x in (2, 3, 4) for y in (2, 3, 4) for z in (2, 3, 4) if 12 <= x * y * z <= 32]
    out = []
    for _ in range(n):
        m = shapes[rng.integers(len(shapes))]
        g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, 3)
        cat = (g[:, None] + fcc).reshape(-1, 3)
        pos = np.concatenate([cat, cat + [0.5, 0, 0]]) * a
        spc = np.concatenate([np.zeros(len(cat), np.int32), np.where(rng.random(len(cat)) < 0.25, 1, 2).astype(np.int32)])
        out.append((pos + rng.normal(0.0, 0.1, size=pos.shape), np.diag([k * a for k in m]), spc))
    return out


def _md_cell(case, rng):
    """A replica of a 256-atom H/O cell (85 water molecules and one H), every copy jittered."""
    L, r = 12.425, case["reps"]
    pos, spc = _molecules(rng, 85, L, extra=1)
    g = np.stack(np.meshgrid(*[np.arange(r)] * 3, indexing="ij"), -1).reshape(-1, 3) * L
    pos = (g[:, None] + pos).reshape(-1, 3)
    pos = pos + rng.normal(0.0, 0.05, size=pos.shape)
    return pos, np.eye(3) * (L * r), np.tile(spc, r ** 3)


SKIN, DT = 0.5, 0.02        # list skin in Angstrom; time step in Angstrom sqrt(amu / eV), about 0.2 fs


def _structures(case, seed):
    rng = np.random.default_rng([seed, 2])
    if case["kind"] == "md":
        return [_md_cell(case, rng)]
    if case["kind"] == "pair":
        n = case["molecules"]
        L = 12.42 * (n / 64.0) ** (1.0 / 3.0)
        pos, spc = _molecules(rng, n, L)
        return [(pos - L * np.floor(pos / L), np.eye(3) * L, spc)]
    if case["basis"] == "water":
        return _water_batch(case, rng)
    if case["basis"] == "lips":
        return _lips_batch(max(case.get("resident", 0), case["structures"]), rng)
    return _argon_batch(case, rng)


def _join(structures):
    n = np.array([len(s[2]) for s in structures])
    return {"natoms": n, "pos": np.concatenate([s[0] for s in structures]), "cells": np.stack([s[1] for s in structures]),
            "species": np.concatenate([s[2] for s in structures]).astype(np.int32)}


# ------------------------------------------------------------------ plain FP64 evaluation


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs_one(pos, cell, rc):
    """(i, j, s) of every pair 0 < |r_i - r_j - s| < rc of one structure, s a lattice vector."""
    n = len(pos)
    inv = torch.linalg.inv(cell)
    frac = pos @ inv.T
    base = torch.floor(frac)
    wide = 1.0 / torch.linalg.norm(inv, dim=1)
    m = [int(math.floor(rc / float(w))) + 1 for w in wide]
    shifts = torch.cartesian_prod(*[torch.arange(-k, k + 1, device=pos.device, dtype=pos.dtype) for k in m])
    wrapped = pos - base @ cell.T
    vec = shifts @ cell.T
    out, step = [], max(1, int(6e7 / (n * n)))
    d0 = wrapped[:, None] - wrapped[None]
    for k in range(0, len(vec), step):
        d = d0[None] - vec[k:k + step, None, None]
        r2 = (d * d).sum(-1)
        q, i, j = torch.nonzero((r2 < rc * rc) & (r2 > 1e-12), as_tuple=True)
        # r_i - r_j - s in the unwrapped positions: s = R (base_i - base_j + shift)
        out.append((i, j, (base[i] - base[j] + shifts[k + q]) @ cell.T))
    return [torch.cat(x) for x in zip(*out)]


def _pairs_grid(pos, L, rc):
    """The same for a large cubic cell, by bins at least rc wide."""
    nb = int(L / rc)
    n, dev = len(pos), pos.device
    base = torch.floor(pos / L)
    w = pos - base * L
    b = (w / L * nb).long().clamp_(0, nb - 1)
    key = (b[:, 0] * nb + b[:, 1]) * nb + b[:, 2]
    order = torch.argsort(key)
    count = torch.bincount(key, minlength=nb ** 3)
    start = torch.cumsum(count, 0) - count
    most = int(count.max())
    slot = torch.arange(n, device=dev) - start[key[order]]
    table = torch.full((nb ** 3, most), -1, device=dev, dtype=torch.long)
    table[key[order], slot] = order
    cells = torch.arange(nb ** 3, device=dev)
    c3 = torch.stack([cells // (nb * nb), cells // nb % nb, cells % nb], 1)
    out = []
    for o in torch.cartesian_prod(*[torch.arange(-1, 2, device=dev)] * 3):
        other = c3 + o
        shift = torch.div(other, nb, rounding_mode="floor")
        oc = other - shift * nb
        oc = (oc[:, 0] * nb + oc[:, 1]) * nb + oc[:, 2]
        step = max(1, int(6e7 / (most * most)))
        for k in range(0, nb ** 3, step):
            ti, tj = table[k:k + step], table[oc[k:k + step]]
            d = w[ti.clamp(min=0)][:, :, None] - (w[tj.clamp(min=0)] + shift[k:k + step, None] * L)[:, None]
            ok = ((d * d).sum(-1) < rc * rc) & (ti >= 0)[:, :, None] & (tj >= 0)[:, None]
            ok &= ti[:, :, None] != tj[:, None]
            c, x, y = torch.nonzero(ok, as_tuple=True)
            i, j = ti[c, x], tj[c, y]
            out.append((i, j, (base[i] - base[j] + shift[k + c]) * L))
    return [torch.cat(x) for x in zip(*out)]


def _pairs(batch, rc):
    """All pairs of a joined batch, sorted by the first atom."""
    dev = _device()
    pos = torch.as_tensor(batch["pos"], device=dev)
    off, got = np.concatenate([[0], np.cumsum(batch["natoms"])]), []
    for s in range(len(batch["natoms"])):
        p, cell = pos[off[s]:off[s + 1]], torch.as_tensor(batch["cells"][s], device=dev)
        i, j, v = _pairs_grid(p, float(cell[0, 0]), rc) if len(p) > 6000 else _pairs_one(p, cell, rc)
        got.append((i + int(off[s]), j + int(off[s]), v))
    i, j, v = (torch.cat(x) for x in zip(*got))
    order = torch.argsort(i, stable=True)
    return i[order], j[order], v[order]


def _monomials(Z):
    ex = [(a, b, m - a - b) for m in range(Z + 1) for a in range(m, -1, -1) for b in range(m - a, -1, -1)]
    f = math.factorial
    return ex, [f(a + b + c) // (f(a) * f(b) * f(c)) for a, b, c in ex]


def _inputs(pot, d, near, sp):
    """Symmetry functions of n centres: d [n, M, 3] displacements, near [n, M] which entries count, sp [n, M]."""
    dev, S = d.device, len(pot["species"])
    t = lambda x: torch.as_tensor(np.asarray(x, dtype=np.float64), device=dev)  # noqa: E731
    r = torch.sqrt((d * d).sum(-1))
    inside = near & (r < RC)
    x = torch.where(inside, r, torch.ones_like(r))
    fc = torch.tanh(1.0 - x / RC) ** 3 if pot["cut"] == "TANH" else 0.5 * (torch.cos(math.pi * x / RC) + 1.0)
    fc = torch.where(inside, fc, torch.zeros_like(fc))
    hot = torch.nn.functional.one_hot(sp, S).to(d.dtype)                        # [n, M, S]
    R = torch.exp(-(t(pot["reta"]) * (x[..., None] - t(pot["rs"]))) ** 2) * fc[..., None]
    rad = torch.bmm(hot.transpose(1, 2).contiguous(), R)                        # [n, S, nr]
    widths = np.unique(pot["aeta"])
    e = torch.exp(-(x[..., None] / t(widths)) ** 2) * fc[..., None]             # [n, M, U]
    U, Z = len(widths), int(max(pot["zeta"]))
    ex, weight = _monomials(Z)
    h = d / x[..., None]
    pw = [torch.ones_like(h)]
    for _ in range(Z):
        pw.append(pw[-1] * h)
    mono = torch.stack([pw[a][..., 0] * pw[b][..., 1] * pw[c][..., 2] for a, b, c in ex], -1)   # [n, M, A]
    eh = (hot[..., None] * e[..., None, :]).reshape(*x.shape, S * U)
    T = torch.bmm(eh.transpose(1, 2).contiguous(), mono).reshape(-1, S, U, len(ex))
    D = (eh * e.repeat(1, 1, S)).sum(1).reshape(-1, S, U)
    degree = np.array([sum(q) for q in ex])
    wd = t(weight)[:, None] * t(degree[:, None] == np.arange(Z + 1)[None])      # [A, Z + 1]
    coef = np.zeros((len(pot["zeta"]), Z + 1))
    for f, (z, lam) in enumerate(zip(pot["zeta"], pot["lam"])):
        for m in range(int(z) + 1):
            coef[f, m] = math.comb(int(z), m) * 0.5 ** int(z) * float(lam) ** m
    which, blocks = torch.as_tensor(np.searchsorted(widths, pot["aeta"]), device=dev), [rad.reshape(len(d), -1)]
    for c in range(S):
        for b in range(c + 1):
            A = (T[:, b] * T[:, c]) @ wd                                       # [n, U, Z + 1]
            if b == c:
                A = 0.5 * (A - D[:, b, :, None])
            blocks.append((A[:, which] * t(coef)).sum(-1))
    return torch.cat(blocks, 1)


def _net(pot, layers, a, G):
    x = torch.as_tensor(pot["inpw"][a], device=G.device) * (G + torch.as_tensor(pot["inpb"][a], device=G.device))
    for k, (w, b) in enumerate(layers):
        x = x @ w.T + b
        if k < len(layers) - 1:
            x = torch.tanh(x) if pot["neuron"] == "TANH" else torch.nn.functional.softplus(x) - math.log(2.0)
    return x[:, 0]


def _tensors(pot):
    return [[(torch.as_tensor(w, device=_device()), torch.as_tensor(b, device=_device())) for w, b in net]
            for net in pot["layers"]]


def _padded(n0, n1, pairs, pos, species):
    """Rows of the centres n0 .. n1-1: displacements, which entries count, species, partners."""
    i, j, v = pairs
    lo, hi = (int(x) for x in torch.searchsorted(i, torch.tensor([n0, n1], device=i.device)))
    ii, jj = i[lo:hi] - n0, j[lo:hi]
    count = torch.bincount(ii, minlength=n1 - n0)
    start = torch.cumsum(count, 0) - count
    M = max(1, int(count.max()))
    slot = torch.arange(hi - lo, device=i.device) - start[ii]
    d = torch.ones((n1 - n0, M, 3), dtype=pos.dtype, device=i.device)
    d[ii, slot] = pos[i[lo:hi]] - pos[jj] - v[lo:hi]
    near = torch.zeros((n1 - n0, M), dtype=torch.bool, device=i.device)
    near[ii, slot] = True
    sp = torch.zeros((n1 - n0, M), dtype=torch.long, device=i.device)
    sp[ii, slot] = species[jj]
    partner = torch.zeros((n1 - n0, M), dtype=torch.long, device=i.device)
    partner[ii, slot] = jj
    return d, near, sp, partner


def _chunk_atoms(pot, n):
    cost = len(pot["species"]) * len(np.unique(pot["aeta"])) + 3 * len(_monomials(int(max(pot["zeta"])))[0])
    return max(256, int(2.5e9 / (8 * cost * 140)))


def _energy_forces(pot, batch, pairs, pos=None, forces=True):
    """(E per structure without vacuum energies, F, per-atom energies, virial per structure)."""
    dev = _device()
    pos = torch.as_tensor(batch["pos"], device=dev) if pos is None else pos
    species = torch.as_tensor(batch["species"], device=dev).long()
    N, layers = len(pos), _tensors(pot)
    F, Ea = torch.zeros_like(pos), torch.zeros(N, dtype=pos.dtype, device=dev)
    S = len(batch["natoms"])
    sof = torch.as_tensor(np.repeat(np.arange(S), batch["natoms"]), device=dev)
    V = torch.zeros((S, 3, 3), dtype=pos.dtype, device=dev)
    step = _chunk_atoms(pot, N)
    for n0 in range(0, N, step):
        n1 = min(N, n0 + step)
        d, near, sp, partner = _padded(n0, n1, pairs, pos, species)
        d.requires_grad_(forces)
        G = _inputs(pot, d, near, sp)
        e = torch.zeros(n1 - n0, dtype=pos.dtype, device=dev)
        for a in range(len(layers)):
            at = torch.nonzero(species[n0:n1] == a)[:, 0]
            if len(at):
                e = e.index_put((at,), _net(pot, layers[a], a, G[at]))
        Ea[n0:n1] = e.detach()
        if forces:
            P, = torch.autograd.grad(e.sum(), d)
            P = torch.where(near[..., None], P, torch.zeros_like(P))
            F[n0:n1] -= P.sum(1)
            F.index_add_(0, partner.reshape(-1), P.reshape(-1, 3))
            V.index_add_(0, sof[n0:n1], -torch.einsum("nmx,nmy->nxy", P, d.detach()))
    E = torch.zeros(S, dtype=pos.dtype, device=dev).index_add_(0, sof, Ea)
    return E, F, Ea, V


def _standardise(pot, batch, pairs):
    """Input bias -mean and scale 1/deviation of every species and input over the batch."""
    pos = torch.as_tensor(batch["pos"], device=_device())
    species = torch.as_tensor(batch["species"], device=_device()).long()
    G, step = [], _chunk_atoms(pot, len(pos))
    for n0 in range(0, len(pos), step):
        n1 = min(len(pos), n0 + step)
        G.append(_inputs(pot, *_padded(n0, n1, pairs, pos, species)[:3]))
    G = torch.cat(G)
    for a in range(len(pot["species"])):
        g = G[species == a]
        dev = g.std(0, unbiased=True)
        pot["inpb"][a] = -g.mean(0).cpu().numpy()
        pot["inpw"][a] = torch.where(dev > 0, 1.0 / dev, torch.ones_like(dev)).cpu().numpy()


def _training_set(case, seed):
    """Potential, structures and labels (a second potential's energies and forces)."""
    batch = _join(_structures(case, seed))
    pairs = _pairs(batch, RC)
    E, F, _, _ = _energy_forces(_potential(case["basis"], seed + 7919), batch, pairs)
    return batch, pairs, E.cpu().numpy(), F.cpu().numpy()


def _draws(case, seed):
    rng = np.random.default_rng([seed, 3])
    return [np.sort(rng.choice(case["resident"], size=case["structures"], replace=False)) for _ in range(16)]


def _pair_frames(case, seed, pos):
    """Positions of the calls of a pair case: atoms drift a little on every call."""
    rng = np.random.default_rng([seed, 4])
    vel = np.clip(rng.normal(0.0, 0.004, size=pos.shape), -0.012, 0.012)
    return [pos + k * vel for k in range(case["calls"])]


# ------------------------------------------------------------------ what a program does


def prepare(case, seed):
    from ann_amd.batch import ResidentSet
    from ann_amd.configs import Batch
    from ann_amd.gpu import Engine
    pot = _potential(case["basis"], seed)
    if case["kind"] == "train":
        batch, _, E, F = _training_set(case, seed)
        eng = Engine(_model(pot))
        buf = torch.empty(2 + eng.nparams, dtype=torch.float64, device=eng.device)     # loss, then the gradient
        st = {"kind": "train", "eng": eng, "buf": buf, "out": (buf[:2], buf[2:]), "step": 0}
        whole = Batch(batch["natoms"], batch["pos"], batch["cells"], batch["species"])
        if case["resident"] > case["structures"]:
            st["set"], st["draws"] = ResidentSet(whole, E, F), _draws(case, seed)
        else:
            eng.set_batch(whole)
            eng.neighbors()
            st["E"], st["F"] = torch.as_tensor(E, device=eng.device), torch.as_tensor(F, device=eng.device)
        return st
    batch = _join(_structures(case, seed))
    if case.get("scaled"):
        _standardise(pot, batch, _pairs(batch, RC))
    eng = Engine(_model(pot))
    if case["kind"] == "pair":
        L, loc, n = float(batch["cells"][0, 0, 0]), batch["pos"], len(batch["pos"])
        g = np.stack(np.meshgrid(*[np.arange(-1, 2)] * 3, indexing="ij"), -1).reshape(-1, 3)
        g = g[np.any(g != 0, axis=1)] * L
        ghost = (g[:, None] + loc).reshape(-1, 3)
        keep = np.all((ghost > -RC - SKIN) & (ghost < L + RC + SKIN), axis=1)
        owner = np.tile(np.arange(n, dtype=np.int32), len(g))[keep]
        offset = np.repeat(g, n, axis=0)[keep]
        x = torch.as_tensor(np.concatenate([loc, ghost[keep]]), device=eng.device)
        r = torch.cdist(x[:n], x, compute_mode="donot_use_mm_for_euclid_dist")
        near = ((r < RC + SKIN) & (r > 0)).cpu().numpy()
        rows = [np.nonzero(row)[0].astype(np.int32) for row in near]
        frames = [np.concatenate([p, p[owner] + offset]) for p in _pair_frames(case, seed, loc)]
        return {"kind": "pair", "eng": eng, "frames": frames, "rows": rows, "owner": owner, "n": n,
                "cell": batch["cells"][0], "species": batch["species"]}
    eng.set_batch(Batch(batch["natoms"], batch["pos"], batch["cells"], batch["species"]))
    dev, S, N = eng.device, len(batch["natoms"]), len(batch["pos"])
    new = lambda *s: torch.empty(s, dtype=torch.float64, device=dev)  # noqa: E731
    if case["kind"] == "md":
        eng.neighbors(RC + SKIN)
        E, F = new(1), new(N, 3)
        eng.energy_forces(out=(E, F, None))
        mass = np.array(pot["mass"])[batch["species"]]
        rng = np.random.default_rng([seed, 5])
        vel = rng.normal(size=(N, 3)) * np.sqrt(8.617333262e-5 * 300.0 / mass)[:, None]
        vel -= (mass[:, None] * vel).sum(0) / mass.sum()
        return {"kind": "md", "eng": eng, "pos0": eng.d_pos.clone(), "F0": F.clone(), "E": E, "F": F,
                "vel0": torch.as_tensor(vel, device=dev), "vel": new(N, 3), "mass": torch.as_tensor(mass, device=dev),
                "steps": case["steps"]}
    # one structure: energy and forces; a batch: also the virials
    return {"kind": case["kind"], "eng": eng, "out": (new(S), new(N, 3), new(S, 3, 3) if S > 1 else None)}


def run(state):
    eng = state["eng"]
    if state["kind"] == "ef":
        eng.neighbors()
        return [x for x in eng.energy_forces(out=state["out"]) if x is not None]
    if state["kind"] == "energies":
        eng.neighbors()
        return [eng.energies(with_evac=False, out=state["out"][0])]
    if state["kind"] == "train":
        if "set" in state:
            b = state["set"].gather(state["draws"][state["step"] % len(state["draws"])], device_meta=False)
            state["step"] += 1
            eng.set_batch_host(b["atom_off"], b["pos"], b["cells_host"], b["species_host"])
            eng.neighbors()
            state["hold"] = b
            eng.train_step(b["energy"], b["forces"], 1.0, 0.1, 1e-3, out=state["out"])
        else:
            eng.train_step(state["E"], state["F"], 1.0, 0.1, 1e-3, out=state["out"])
        return [state["buf"]]
    if state["kind"] == "md":
        # the segment starts from the same positions and velocities on every pass
        eng.d_pos.copy_(state["pos0"])
        state["vel"].copy_(state["vel0"])
        state["F"].copy_(state["F0"])
        eng.neighbors(RC + SKIN)
        for _ in range(state["steps"]):
            eng.md_step(DT, state["mass"], state["vel"], state["F"], E=state["E"])
        return [eng.d_pos, state["vel"], state["F"], state["E"]]
    sums, F, Ea = [], [], []
    for k, x in enumerate(state["frames"]):
        e, f, ea, vir = eng.pair_compute(x, state["species"], state["cell"], state["owner"],
                                         state["rows"] if k == 0 else None, RC + SKIN, state["n"], new_list=k == 0)
        sums.append(np.concatenate([[e], vir]))     # the seven global sums a host code keeps
        F.append(f)
        Ea.append(ea)
    return [np.stack(sums), np.stack(F), np.stack(Ea)]


# ------------------------------------------------------------------ sizes and FP64 results


def work(case):
    """Bytes: positions, species, cells and labels read, results written, once.  Operations: per pair in
    range the radial functions and the sums over the monomials of the unit vector (the triplet sums'
    exact factorisation; above exponent 5 the triplets themselves), per atom the network forward and
    backward (and twice more for a training step's second backward and gradient)."""
    b = _basis(case["basis"])
    S, nr, na = len(b["species"]), len(b["rs"]), len(b["aeta"])
    nin = S * nr + S * (S + 1) // 2 * na
    mac, prev = 0, nin
    for h in b["hidden"] + [1]:
        mac, prev = mac + prev * h, h
    U, Z = len(np.unique(b["aeta"])), int(max(b["zeta"]))
    M = (Z + 1) * (Z + 2) * (Z + 3) // 6
    if case["kind"] == "md":
        N, n, times = 256 * case["reps"] ** 3, 121, case["steps"]
    elif case["kind"] == "pair":
        N, n, times = 3 * case["molecules"], 91, case["calls"]
    elif case["basis"] == "water":
        N, n, times = 3 * case["molecules"] * case["structures"], 91 if not case["uneven"] else 82, 1
    elif case["basis"] == "lips":
        N, n, times = 180 * case["structures"], 41, 1
    else:
        N, n, times = 4 * case["cells"] ** 3 * case["structures"], 18, 1
    angular = n * M * (2 + 2 * U) if Z <= 5 else n * (n - 1) / 2 * (8 + 4 * na)
    one = n * (10 + 6 * nr) + angular + 2 * mac
    if case["kind"] != "energies":
        one += n * (20 + 6 * nr) + (n * M * (4 * U + 16) if Z <= 5 else n * (n - 1) / 2 * (52 + 8 * na)) + 2 * mac
    if case["kind"] == "train":
        one += n * (20 + 8 * nr) + n * M * (9 + 6 * U) + 12 * mac
    per = {"ef": 24 + 4 + 24, "energies": 24 + 4, "train": 24 + 4 + 24, "md": 24 + 4 + 8 + 24 + 24 + 72, "pair": 24 + 32}
    return {"bytes": float(N * per[case["kind"]] * (times if case["kind"] == "pair" else 1)), "flops": float(N * one * times)}


def exact(case, seed):
    pot = _potential(case["basis"], seed)
    evac = np.array(pot["evac"])
    if case["kind"] == "train":
        batch, pairs, Eref, Fref = _training_set(case, seed)
        n = batch["natoms"]
        off = np.concatenate([[0], np.cumsum(n)])
        pick = _draws(case, seed)[0] if case["resident"] > case["structures"] else np.arange(case["structures"])
        return [_train_exact(pot, batch, pairs, Eref, Fref, off, pick)]
    batch = _join(_structures(case, seed))
    S = len(batch["natoms"])
    sof = np.repeat(np.arange(S), batch["natoms"])
    vac = np.bincount(sof, evac[batch["species"]], minlength=S)
    pairs = _pairs(batch, RC + SKIN if case["kind"] in ("md", "pair") else RC)
    if case["kind"] == "md":
        return _md_exact(case, seed, pot, batch, pairs, vac)
    if case["kind"] == "pair":
        sums, Fs, Eas = [], [], []
        for x in _pair_frames(case, seed, batch["pos"]):
            E, F, Ea, V = _energy_forces(pot, batch, pairs, torch.as_tensor(x, device=_device()))
            V = V[0].cpu().numpy()
            sums.append(np.concatenate([E.cpu().numpy() + vac, V[[0, 1, 2, 0, 0, 1], [0, 1, 2, 1, 2, 2]]]))
            Fs.append(F.cpu().numpy())
            Eas.append(Ea.cpu().numpy() + evac[batch["species"]])
        return [np.stack(sums), np.stack(Fs), np.stack(Eas)]
    if case.get("scaled"):
        _standardise(pot, batch, pairs)
    E, F, _, V = _energy_forces(pot, batch, pairs, forces=case["kind"] == "ef")
    if case["kind"] == "energies":
        return [E]
    E = E + torch.as_tensor(vac, device=E.device)
    return [E, F, V] if S > 1 else [E, F]


def _md_exact(case, seed, pot, batch, pairs, vac):
    dev = _device()
    pos = torch.as_tensor(batch["pos"], device=dev)
    mass = np.array(pot["mass"])[batch["species"]]
    rng = np.random.default_rng([seed, 5])
    vel = rng.normal(size=pos.shape) * np.sqrt(8.617333262e-5 * 300.0 / mass)[:, None]
    vel -= (mass[:, None] * vel).sum(0) / mass.sum()
    vel, m = torch.as_tensor(vel, device=dev), torch.as_tensor(mass, device=dev)[:, None]
    E, F, _, _ = _energy_forces(pot, batch, pairs, pos)
    for _ in range(case["steps"]):
        vel = vel + 0.5 * DT * F / m
        pos = pos + DT * vel
        E, F, _, _ = _energy_forces(pot, batch, pairs, pos)
        vel = vel + 0.5 * DT * F / m
    return [pos, vel, F, E + torch.as_tensor(vac, device=dev)]


def _train_exact(pot, batch, pairs, Eref, Fref, off, pick):
    """[energy loss, force loss, gradient] of the drawn structures, by double differentiation."""
    dev, B = _device(), len(pick)
    layers = [[(w.clone().requires_grad_(), b.clone().requires_grad_()) for w, b in net] for net in _tensors(pot)]
    params = [p for net in layers for p in [b for _, b in net] + [w for w, _ in net]]
    grad = [torch.zeros_like(p) for p in params]
    pos = torch.as_tensor(batch["pos"], device=dev)
    species = torch.as_tensor(batch["species"], device=dev).long()
    loss = torch.zeros(2, dtype=pos.dtype, device=dev)
    Eref, Fref = torch.as_tensor(Eref, device=dev), torch.as_tensor(Fref, device=dev)
    for s in pick:
        n0, n1 = int(off[s]), int(off[s + 1])
        n = n1 - n0
        d, near, sp, partner = _padded(n0, n1, pairs, pos, species)
        d.requires_grad_()
        G = _inputs(pot, d, near, sp)
        e = torch.zeros(n, dtype=pos.dtype, device=dev)
        for a in range(len(layers)):
            at = torch.nonzero(species[n0:n1] == a)[:, 0]
            if len(at):
                e = e.index_put((at,), _net(pot, layers[a], a, G[at]))
        P, = torch.autograd.grad(e.sum(), d, create_graph=True)
        P = torch.where(near[..., None], P, torch.zeros_like(P))
        F = torch.zeros((n, 3), dtype=pos.dtype, device=dev).index_add(0, (partner - n0).clamp(min=0).reshape(-1),
                                                                       P.reshape(-1, 3)) - P.sum(1)
        lE = 0.5 * ((e.sum() - Eref[s]) / n) ** 2 / B
        lF = 0.1 / (3.0 * n) * ((F - Fref[n0:n1]) ** 2).sum() / B
        for q, g in enumerate(torch.autograd.grad(lE + lF, params, allow_unused=True)):
            if g is not None:
                grad[q] += g
        loss += torch.stack([lE.detach(), lF.detach()])
    flat = [g if g.dim() == 1 else g.T.reshape(-1) for g in grad]
    return torch.cat([loss] + flat)
