"""Neighbour lists of structures in which only part of the bins fit the staged
search, bit for bit against the FP64 oracle's list: built, moved and built again
on the same context, so that the fill that runs beside the wait for the list size
meets rows the first search pass left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model():
    from ann_amd import configs
    return configs.model_ar256()


def _slab(L, height, fill, spacing, seed):
    """Atoms on a jittered grid in the lower part of an L x L x height cell, a few above it."""
    from ann_amd import configs
    rng = np.random.default_rng(seed)
    axes = [np.arange(int(x / spacing)) * spacing for x in (L, L, fill)]
    pos = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    pos = pos + rng.normal(0.0, 0.05 * spacing, size=pos.shape)
    gas = rng.uniform([0, 0, fill], [L, L, height], size=(40, 3))
    pos = rng.permutation(np.concatenate([pos, gas]))
    return configs.single(pos, np.diag([L, L, height]), np.zeros(len(pos), np.int32))


def _check(eng, pos, batch, orc, rc):
    nl = eng.nlist()
    ref = orc.nlist(pos, batch.cells[0].reshape(3, 3), batch.species, rc)
    for k in ("off", "idx", "img", "rev"):
        assert np.array_equal(nl[k], getattr(ref, k)), k


# L, height, filled height, spacing, cutoff: a slab whose dense part overflows even the
# smallest search box (atoms above it have short rows), one below and one above the
# largest structure with rank tables; water-like slabs whose mean density admits
# 2 x 2 x 2 bins that the dense part overflows
CASES = [(11.0, 24.0, 10.5, 0.875, 4.0, 4), (13.0, 24.0, 12.0, 0.875, 4.0, 4), (40.0, 40.0, 28.0, 2.15, 7.5, 1),
         (50.0, 50.0, 30.0, 2.15, 8.0, 1)]


@pytest.mark.parametrize("L,height,fill,spacing,rc,wide", CASES)
def test_partly_overflowed_bins(oracle_mod, L, height, fill, spacing, rc, wide):
    import torch
    from ann_amd.gpu import Engine
    model, batch = _model(), _slab(L, height, fill, spacing, 70)
    orc = oracle_mod.Oracle(model)
    eng = Engine(model, "cuda:0")
    eng.set_batch(batch)
    rng = np.random.default_rng(71)
    pos = batch.pos.copy()
    eng.profile(True)
    for step in range(4):                       # the first build allocates, the others fill beside the wait
        eng.neighbors(rc)
        widest = eng.nlist_size()[1]
        _check(eng, pos, batch, orc, rc)
        pos = pos + rng.normal(0.0, 0.02, size=pos.shape)
        eng.d_pos.copy_(torch.from_numpy(pos))
    # 2 x 2 x 2 bins that do not fit are searched one by one, after the first build without a second pass
    assert eng.profile_get("nb_search_wide")[1] == wide
    assert eng.profile_get("nb_search_split")[1] == (4 if wide == 1 else 0)
    print(f"  {batch.ntotal} atoms, rc {rc}: widest row {widest}", flush=True)


@pytest.mark.parametrize("L,spacing,wide", [(80.0, 1.1, 1), (40.0, 1.1, 1), (40.0, 0.85, 4)])
def test_droplet(oracle_mod, L, spacing, wide):
    """A droplet in an otherwise empty cell, with more bins than atoms; its inner bins fit a
    block one by one (rows of 200) or not (rows of 437)."""
    import torch
    from ann_amd import configs
    from ann_amd.gpu import Engine
    rng = np.random.default_rng(74)
    g = np.arange(int(14.5 / spacing)) * spacing
    # around the cell's first two bins per direction (2.05 or 2.1 wide), across its corner
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) - 0.5 * g[-1] + 2.05
    pos = rng.permutation(pos + rng.normal(0.0, 0.05 * spacing, size=pos.shape))
    batch = configs.single(pos, np.eye(3) * L, np.zeros(len(pos), np.int32))
    assert len(pos) < (L // 2.0 - 1) ** 3
    orc, eng = oracle_mod.Oracle(_model()), Engine(_model(), "cuda:0")
    eng.set_batch(batch)
    eng.profile(True)
    for step in range(4):
        eng.neighbors(4.0)
        assert eng.nlist_size()[1] > 0
        _check(eng, pos, batch, orc, 4.0)
        pos = pos + rng.normal(0.0, 0.01, size=pos.shape)
        eng.d_pos.copy_(torch.from_numpy(pos))
    assert eng.profile_get("nb_search_wide")[1] == wide and eng.profile_get("nb_search_split")[1] == 4


@pytest.mark.parametrize("n", [1900, 2600])
def test_refused_then_good(oracle_mod, n):
    """A build refused for rows above the capacity leaves no fault behind for the next one."""
    import torch
    from ann_amd import configs
    from ann_amd.gpu import AnnError, Engine
    L, rc = (n / 0.57) ** (1.0 / 3.0), 5.0
    pos = np.random.default_rng(72).uniform(0, L, size=(n, 3))
    bad = pos.copy()
    bad[-560:] = L / 2 + (pos[-560:] - L / 2) * (2.0 / L)       # 560 atoms within rc of each other, fewer pairs in all
    batch = configs.single(pos, np.eye(3) * L, np.zeros(n, np.int32))
    orc = oracle_mod.Oracle(_model())
    eng = Engine(_model(), "cuda:0")
    eng.set_batch(batch)
    eng.neighbors(rc)
    for _ in range(2):
        eng.d_pos.copy_(torch.from_numpy(bad))
        with pytest.raises(AnnError):
            eng.neighbors(rc)
        eng.d_pos.copy_(torch.from_numpy(pos))
        eng.neighbors(rc)
        _check(eng, pos, batch, orc, rc)


@pytest.mark.parametrize("n,L,rc", [(2, 4.0, 6.0), (301, 16.0, 6.0), (2601, 32.0, 6.0)])
def test_far_from_the_cell(oracle_mod, n, L, rc):
    """A structure moved by whole cells, also past the +-511 that a packed image holds,
    keeps its list.  Coordinates are multiples of 2^-10, so the move is exact."""
    import torch
    from ann_amd import configs
    from ann_amd.gpu import Engine
    rng = np.random.default_rng(73)
    pos = rng.integers(0, int(L * 1024), size=(n, 3)) / 1024.0
    batch = configs.single(pos, np.eye(3) * L, np.zeros(n, np.int32))
    eng = Engine(_model(), "cuda:0")
    eng.set_batch(batch)
    eng.neighbors(rc)
    _check(eng, pos, batch, oracle_mod.Oracle(_model()), rc)
    home = eng.nlist()
    for k in (511, -511, 512, -512, -513, 1000, -1024, 5000):
        for axis in ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)):
            eng.d_pos.copy_(torch.from_numpy(pos + np.array(axis) * (k * L)))
            eng.neighbors(rc)
            away = eng.nlist()
            for q in ("off", "idx", "img", "rev", "geo"):
                assert np.array_equal(away[q], home[q]), (k, axis, q)
