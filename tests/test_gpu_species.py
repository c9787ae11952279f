"""Moment form with four to eight species (G, adjoint, tangent and the FP64 inputs
of the instances that hold every species' sums in registers) against the FP64
oracle: rows of a few and of more than 64 entries, species absent from rows and
from whole structures, grid dispatch and work queues.

Bars (those of the other parity tests): energies <= 1e-6 eV/atom, forces,
virial and tangent relative RMS <= 1e-5, G <= 2e-5 of the row maximum, FP64 G
<= 1e-10 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(S, z, nr):
    from ann_amd.model import ANG, CUT, NEURON, RAD, Model, init_network
    rng = np.random.default_rng(400 + 10 * S + z)
    rs = np.linspace(0.8, 5.5, nr)
    rad = (RAD["GAUSSIAN"], rs, np.full(nr, 1.0 / (rs[1] - rs[0])))
    widths = [1.5, 3.0] if S == 4 else [2.5]
    ang = (ANG["GAUSS"], np.repeat(widths, 2), np.full(2 * len(widths), float(z)), np.tile([1, -1], len(widths)))
    npair = S * (S + 1) // 2
    nets = [init_network(S * nr + npair * 2 * len(widths), [16, 12], NEURON["TANH"], rng) for _ in range(S)]
    return Model([f"X{a}" for a in range(S)], np.ones(S), np.zeros(S), 6.0, CUT["TANH"],
                 [[rad] * S for _ in range(S)], [[ang] * npair for _ in range(S)], nets)


def _batch(S):
    """Water density, a sparse gas, one atom of the last species among the first, one atom alone."""
    from ann_amd import configs
    from ann_amd.configs import Batch
    rng = np.random.default_rng(S)

    def grid(n, L, species):
        g = int(np.ceil(n ** (1 / 3)))
        site = rng.permutation(g ** 3)[:n]
        p = (np.stack([site // (g * g), site // g % g, site % g], 1) + 0.5) * (L / g)
        return configs.single(p + rng.normal(0.0, 0.1 * L / g, size=(n, 3)), np.eye(3) * L, species.astype(np.int32))
    lone = np.zeros(60)
    lone[7] = S - 1
    return Batch.concat([grid(150, 11.4, rng.integers(0, S, 150)), grid(70, 16.0, rng.integers(0, S, 70)),
                         grid(60, 9.0, lone), grid(40, 8.0, rng.integers(0, 2, 40) * (S - 1)),
                         configs.single(np.zeros((1, 3)), np.eye(3) * 20.0, np.array([S - 1], np.int32))])


@pytest.mark.parametrize("S,z,nr", [(4, 1, 8), (4, 2, 8), (4, 3, 8), (4, 4, 8), (4, 5, 8), (5, 2, 5), (6, 4, 5),
                                    (8, 1, 4), (8, 2, 4), (8, 5, 4)])
def test_many_species(oracle_mod, S, z, nr):
    import torch
    from ann_amd.gpu import FAST, Engine
    model, batch = _model(S, z, nr), _batch(S)
    orc = oracle_mod.Oracle(model)
    Eo, Fo, Vo = orc.compute_batch(batch, nthreads=4)
    u = np.random.default_rng(45).normal(size=(batch.ntotal, 3))
    ref = []
    for k in range(batch.nstruc):
        pos, cell, sp = batch.struc(k)
        ref.append((orc.symm(pos, cell, sp), orc.tangent(pos, cell, sp, u[batch.atom_off[k]:batch.atom_off[k + 1]])))
    for queue in (0, 1):
        eng = Engine(model, "cuda:0")
        eng.set_tuning([4, 4, 1, 0, 0, queue])
        eng.set_batch(batch)
        eng.neighbors()
        assert eng.nlist_size()[1] > 64
        ud = torch.tensor(u, device="cuda:0")
        v0 = eng.tangent(ud, FAST).cpu().numpy()            # no moments of this list are stored yet
        eng.profile(True)
        E, F, V = (x.cpu().numpy() for x in eng.energy_forces(FAST))
        assert eng.profile_get("symm_fwd_mom")[1] == 1 and eng.profile_get("symm_bwd_mom")[1] == 1
        eng.profile(False)
        eF = np.linalg.norm(F - Fo) / np.linalg.norm(Fo)
        eV = np.linalg.norm(V.reshape(-1) - np.asarray(Vo).reshape(-1)) / np.linalg.norm(Vo)
        eE = np.max(np.abs(E - Eo) / batch.natoms)
        G = eng.symm(FAST).cpu().numpy().astype(np.float64)
        v = eng.tangent(ud, FAST).cpu().numpy()
        eng.set_precise_ratio(-1.0)
        G64 = eng.symm64().cpu().numpy()
        off, eG, eG64, eT, eT0 = batch.atom_off, 0.0, 0.0, 0.0, 0.0
        for k, (Go, vr) in enumerate(ref):
            n, s = Go.shape[1], slice(off[k], off[k + 1])
            top = np.maximum(np.abs(Go).max(axis=1, keepdims=True), 1e-30)
            eG = max(eG, float(np.max(np.abs(G[s, :n] - Go) / top)))
            eG64 = max(eG64, float(np.max(np.abs(G64[s, :n] - Go) / top)))
            scale = max(np.linalg.norm(vr), 1e-30)
            eT = max(eT, float(np.linalg.norm(v[s, :n] - vr) / scale))
            eT0 = max(eT0, float(np.linalg.norm(v0[s, :n] - vr) / scale))
        print(f"  S {S} z {z} queue {queue}: E {eE:.1e} F {eF:.1e} V {eV:.1e} G {eG:.1e} G64 {eG64:.1e} "
              f"tangent {eT:.1e} {eT0:.1e}", flush=True)
        assert eE <= 1e-6 and eF <= 1e-5 and eV <= 1e-5 and eG <= 2e-5 and eG64 <= 1e-10 and eT <= 1e-5 and eT0 <= 1e-5


# widest rows around the function rows held in LDS at a time (4, 8, 24, 32)
@pytest.mark.parametrize("z", [2, 4])
@pytest.mark.parametrize("n", [1, 4, 5, 6, 9, 25, 26, 33, 34])
def test_short_rows(oracle_mod, n, z):
    """n atoms within one cutoff of each other (rows of n - 1), twice, and a lone atom."""
    import torch
    from ann_amd import configs
    from ann_amd.configs import Batch
    from ann_amd.gpu import FAST, Engine
    rng = np.random.default_rng(500 + n)
    g = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3)
    def one(k):
        p = g[rng.permutation(64)[:k]] * 1.1 + rng.normal(0.0, 0.08, size=(k, 3))
        return configs.single(p, np.eye(3) * 30.0, rng.integers(0, 4, k).astype(np.int32))
    batch = Batch.concat([one(n), one(1), one(n)])
    model = _model(4, z, 8)
    orc, eng = oracle_mod.Oracle(model), Engine(model, "cuda:0")
    eng.set_batch(batch)
    eng.neighbors()
    assert eng.nlist_size()[1] == n - 1
    u = rng.normal(size=(batch.ntotal, 3))
    eng.energy_forces(FAST)
    v = eng.tangent(torch.tensor(u, device="cuda:0"), FAST).cpu().numpy()
    G = eng.symm(FAST).cpu().numpy().astype(np.float64)
    for k in range(batch.nstruc):
        pos, cell, sp = batch.struc(k)
        s = slice(batch.atom_off[k], batch.atom_off[k + 1])
        Go, vr = orc.symm(pos, cell, sp), orc.tangent(pos, cell, sp, u[s])
        m = Go.shape[1]
        assert np.max(np.abs(G[s, :m] - Go)) <= 2e-5 * max(np.abs(Go).max(), 1e-30)
        assert np.linalg.norm(v[s, :m] - vr) <= 1e-5 * np.linalg.norm(vr)
