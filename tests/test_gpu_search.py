"""The staged neighbour search where its candidate sort and blocking change, bit
for bit against the FP64 oracle's list: structures below and above 1,024 atoms
(one and several atom indices per bucket) with atoms in random order, single-bin
and super-bin blocks, chunks of candidates that are and are not full, rows of
more than 256 neighbours, several images of one partner, and a build in which a
position is not finite followed by a good one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(rc=6.0):
    from ann_amd import configs
    m = configs.model_ar256()
    m.rc = rc
    return m


def _gas(n, L, seed):
    from ann_amd import configs
    rng = np.random.default_rng(seed)
    return configs.single(rng.uniform(-L, 2 * L, size=(n, 3)), np.eye(3) * L, np.zeros(n, np.int32))


def _check(eng, batch, orc, rc):
    nl, off = eng.nlist(), batch.atom_off
    for k in range(batch.nstruc):
        ref = orc.nlist(*batch.struc(k), rc)
        s0, s1 = nl["off"][off[k]], nl["off"][off[k + 1]]
        assert np.array_equal(nl["off"][off[k]:off[k + 1] + 1] - s0, ref.off)
        assert np.array_equal(nl["idx"][s0:s1] - off[k], ref.idx)
        assert np.array_equal(nl["img"][s0:s1], ref.img)
        assert np.array_equal(nl["rev"][s0:s1] - s0, ref.rev)


# atoms, box, cutoff, copies: dense rows (352 neighbours on average, up to about 400),
# small cells with several images per partner, index ranges of 1,023 to 5,000
CASES = [(1, 9.0, 6.0, 1), (2, 4.5, 6.0, 5), (63, 9.0, 5.0, 3), (64, 9.0, 5.0, 80), (65, 9.0, 5.0, 3),
         (700, 12.0, 6.0, 1), (1023, 22.0, 6.0, 2), (1025, 22.0, 6.0, 12), (2049, 30.0, 6.5, 1), (5000, 40.0, 6.0, 1)]


@pytest.mark.parametrize("n,L,rc,copies", CASES)
def test_list_bit_exact(oracle_mod, n, L, rc, copies):
    from ann_amd.configs import Batch
    from ann_amd.gpu import Engine
    model = _model()
    batch = Batch.concat([_gas(n, L, 50 + c) for c in range(copies)])
    eng = Engine(model, "cuda:0")
    orc = oracle_mod.Oracle(model)
    for single in (0, 1):
        eng.set_tuning([4, 4, 1, 0, single])
        eng.set_batch(batch)
        eng.neighbors(rc)
        _check(eng, batch, orc, rc)
    print(f"  {n} x {copies}: widest row {eng.nlist_size()[1]}", flush=True)
    if n == 700:
        assert eng.nlist_size()[1] > 256


def test_nonfinite_then_good(oracle_mod):
    from ann_amd.gpu import AnnError, Engine
    model, batch = _model(), _gas(65, 9.0, 60)
    eng = Engine(model, "cuda:0")
    for bad in (np.inf, -np.inf, np.nan, 1e300):
        pos = batch.pos.copy()
        pos[17, 2] = bad
        eng.set_batch(type(batch)(batch.natoms, pos, batch.cells, batch.species))
        with pytest.raises(AnnError):
            eng.neighbors(5.0)
    eng.set_batch(batch)
    eng.neighbors(5.0)
    _check(eng, batch, oracle_mod.Oracle(model), 5.0)


# atoms, box, cutoff, copies around the rule for rank tables: structures of 63 and 64
# atoms, the cutoff sphere 0.84 and 0.86 of the cell, small cells with many images of
# a partner; and a batch whose pairs are half in either kind
@pytest.mark.parametrize("n,L,rc,copies", [(63, 12.0, 6.0, 4), (64, 12.0, 6.0, 4), (64, (905.0 / 0.84) ** (1 / 3), 6.0, 3),
                                           (64, (905.0 / 0.86) ** (1 / 3), 6.0, 3), (32, 6.8, 6.0, 4), (96, 9.9, 6.0, 3)])
def test_rank_table_rule(oracle_mod, n, L, rc, copies):
    from ann_amd.configs import Batch
    from ann_amd.gpu import Engine
    eng, orc = Engine(_model(), "cuda:0"), oracle_mod.Oracle(_model())
    same = Batch.concat([_gas(n, L, 80 + c) for c in range(copies)])
    mixed = Batch.concat([same, _gas(200, 14.0, 90), _gas(3, 9.0, 91)])
    for batch in (same, mixed, same):
        eng.set_batch(batch)
        eng.neighbors(rc)
        _check(eng, batch, orc, rc)


# the largest structure among many: up to 256 atoms and 216 bins a structure is binned
# by one wavefront, 257 atoms or 343 bins take eight
@pytest.mark.parametrize("n,L", [(2, 9.0), (255, 20.0), (256, 20.0), (257, 20.0), (200, 21.5)])
def test_many_structures(oracle_mod, n, L):
    from ann_amd.configs import Batch
    from ann_amd.gpu import Engine
    eng, orc = Engine(_model(), "cuda:0"), oracle_mod.Oracle(_model())
    batch = Batch.concat([_gas(1 + c % 5, 8.0 + 0.5 * (c % 3), 100 + c) for c in range(1540)] + [_gas(n, L, 99)])
    for _ in range(2):
        eng.set_batch(batch)
        eng.neighbors(6.0)
        _check(eng, batch, orc, 6.0)


@pytest.mark.parametrize("n", [65, 2100])
def test_nonfinite_between_good(oracle_mod, n):
    """The same on a context whose list arrays are there, so that the fill beside the
    wait also runs on the bad build; the next builds and the size report stand."""
    import torch
    from ann_amd.gpu import AnnError, Engine
    model, batch = _model(), _gas(n, 9.0 if n < 100 else 28.0, 61)
    eng, orc = Engine(model, "cuda:0"), oracle_mod.Oracle(model)
    eng.set_batch(batch)
    eng.neighbors(5.0)
    _check(eng, batch, orc, 5.0)
    for bad in (np.inf, np.nan, 1e300):
        eng.d_pos[17, 2] = bad
        with pytest.raises(AnnError):
            eng.neighbors(5.0)
        eng.d_pos.copy_(torch.from_numpy(batch.pos))
        for _ in range(2):
            eng.neighbors(5.0)
            assert eng.nlist_size()[1] > 0
        _check(eng, batch, orc, 5.0)
