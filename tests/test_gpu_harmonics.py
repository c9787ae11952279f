"""The moment form at every degree bound (largest zeta 1 to 5, one compiled
kernel each) against the FP64 oracle: G, energies, forces, virials, the adjoint
with and without stored moments, the tangent, and the FP64 inputs, on one, two
and three species with rows from a few to over a hundred neighbours.

Bars (those of the other parity tests): energies <= 1e-6 eV/atom, forces,
virial and tangent relative RMS <= 1e-5, G <= 2e-5 of the row maximum, FP64 G
<= 1e-10 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(nspecies, z, nr=8):
    from ann_amd.model import ANG, CUT, NEURON, RAD, Model, init_network
    rng = np.random.default_rng(40 + z)
    rs = np.linspace(0.8, 5.5, nr)
    rad = (RAD["GAUSSIAN"], rs, np.full(nr, 1.0 / (rs[1] - rs[0])))
    zz = [float(z)] if z == 1 else [float(z - 1), float(z)]
    eta = np.repeat([1.5, 3.0], 2 * len(zz))
    zeta = np.tile(np.repeat(zz, 2), 2)
    lam = np.tile([1, -1], 2 * len(zz))
    ang = (ANG["GAUSS"], eta, zeta, lam)
    npair = nspecies * (nspecies + 1) // 2
    nin = nspecies * nr + npair * len(eta)
    nets = [init_network(nin, [16, 12], NEURON["TANH"], rng) for _ in range(nspecies)]
    return Model(["A", "B", "C"][:nspecies], np.ones(nspecies), np.zeros(nspecies), 6.0, CUT["TANH"],
                 [[rad] * nspecies for _ in range(nspecies)], [[ang] * npair for _ in range(nspecies)], nets)


def _batch(nspecies):
    from ann_amd import configs
    if nspecies == 1:
        return configs.struc_ar256(seed=41)
    if nspecies == 2:
        return configs.batch_uneven(3, seed=42, nmin=32, nmax=200)
    return configs.batch_lips(3, seed=43)


@pytest.mark.parametrize("nspecies", [1, 2, 3])
@pytest.mark.parametrize("z", [1, 2, 3, 4, 5])
def test_every_degree_bound(oracle_mod, nspecies, z):
    import torch
    from ann_amd.gpu import FAST, Engine
    model, batch = _model(nspecies, z), _batch(nspecies)
    orc = oracle_mod.Oracle(model)
    eng = Engine(model, "cuda:0")
    eng.set_batch(batch)
    eng.neighbors()
    eng.profile(True)
    dE = torch.from_numpy(np.random.default_rng(44).normal(size=(batch.ntotal, eng.ldg)).astype(np.float32)).cuda()
    P0 = eng.symm_bwd(dE).clone()               # no moments of this list are stored yet
    E, F, V = (x.cpu().numpy() for x in eng.energy_forces(FAST))
    assert eng.profile_get("symm_fwd_mom")[1] == 1 and eng.profile_get("symm_bwd_mom")[1] == 2
    P1 = eng.symm_bwd(dE)                       # moments stored by the call before
    eng.profile(False)
    scale = float(P0.double().norm())
    assert float((P0.double() - P1.double()).norm()) <= 1e-5 * scale
    Eo, Fo, Vo = orc.compute_batch(batch, nthreads=4)
    eF = np.linalg.norm(F - Fo) / np.linalg.norm(Fo)
    eV = np.linalg.norm(V.reshape(-1) - np.asarray(Vo).reshape(-1)) / np.linalg.norm(Vo)
    eE = np.max(np.abs(E - Eo) / batch.natoms)
    G = eng.symm(FAST).cpu().numpy().astype(np.float64)
    eng.set_precise_ratio(-1.0)
    G64 = eng.symm64().cpu().numpy()
    u = np.random.default_rng(45).normal(size=(batch.ntotal, 3))
    v = eng.tangent(torch.tensor(u, device="cuda:0"), FAST).cpu().numpy()
    off, eG, eG64, eT = batch.atom_off, 0.0, 0.0, 0.0
    for k in range(batch.nstruc):
        pos, cell, sp = batch.struc(k)
        Go = orc.symm(pos, cell, sp)
        n = Go.shape[1]
        top = np.maximum(np.abs(Go).max(axis=1, keepdims=True), 1e-30)
        eG = max(eG, float(np.max(np.abs(G[off[k]:off[k + 1], :n] - Go) / top)))
        eG64 = max(eG64, float(np.max(np.abs(G64[off[k]:off[k + 1], :n] - Go) / top)))
        vr = orc.tangent(pos, cell, sp, u[off[k]:off[k + 1]])
        eT = max(eT, float(np.linalg.norm(v[off[k]:off[k + 1], :n] - vr) / np.linalg.norm(vr)))
    print(f"  S {nspecies} z {z}: E {eE:.1e} F {eF:.1e} V {eV:.1e} G {eG:.1e} G64 {eG64:.1e} tangent {eT:.1e}", flush=True)
    assert eE <= 1e-6 and eF <= 1e-5 and eV <= 1e-5 and eG <= 2e-5 and eG64 <= 1e-10 and eT <= 1e-5


def test_moments_kept_by_calls_that_move_nothing(oracle_mod):
    """The loss, the structure weights and the tuning leave the stored moments in use
    (the adjoint is then the same bits); new geometry does not."""
    import torch
    from ann_amd import configs
    from ann_amd.gpu import FAST, Engine
    model, batch = configs.model_lips(), configs.batch_lips(3, seed=43)
    eng = Engine(model, "cuda:0")
    eng.set_batch(batch)
    eng.neighbors()
    eng.energy_forces(FAST)
    rng = np.random.default_rng(46)
    dE = torch.from_numpy(rng.normal(size=(batch.ntotal, eng.ldg)).astype(np.float32)).cuda()
    u = torch.from_numpy(rng.normal(size=(batch.ntotal, 3))).cuda()
    P, v = eng.symm_bwd(dE).clone(), eng.tangent(u).clone()
    w = torch.ones(batch.nstruc, dtype=torch.float64, device="cuda:0")
    for call in (lambda: eng.set_loss("HUBER", 0.5), lambda: eng.set_struc_weights(w, w),
                 lambda: eng.set_tuning([4, 4, 1, 0, 0])):
        call()
        assert torch.equal(eng.symm_bwd(dE), P) and torch.equal(eng.tangent(u), v)
    eng.d_pos += 0.01 * u
    eng.refresh_geometry()
    P0, v0 = eng.symm_bwd(dE).clone(), eng.tangent(u).clone()   # sums the moments itself
    assert float((P0 - P).norm()) > 1e-4 * float(P.norm())      # the old moments would give nearly the old values
    eng.energy_forces(FAST)
    for a, b in ((eng.symm_bwd(dE), P0), (eng.tangent(u), v0)):
        assert float((a.double() - b.double()).norm()) <= 1e-5 * float(b.double().norm())


@pytest.mark.parametrize("z", [3, 4, 5])
def test_recomputing_adjoint_of_large_batches(z):
    """More wavefronts than the chip's LDS holds at 64 function rows each (32 from degree 4 on)."""
    import torch
    from ann_amd import configs
    from ann_amd.gpu import FAST, Engine
    eng = Engine(_model(2, z), "cuda:0")
    eng.set_batch(configs.batch_water(32, seed=47))
    eng.neighbors()
    dE = torch.from_numpy(np.random.default_rng(48).normal(size=(eng.N, eng.ldg)).astype(np.float32)).cuda()
    P0 = eng.symm_bwd(dE).double()              # no moments of this list are stored yet
    eng.energy_forces(FAST)
    assert float((eng.symm_bwd(dE).double() - P0).norm()) <= 1e-5 * float(P0.norm())
