"""The order in which a step deals workgroups to the XCDs, beyond the size of
the last-level cache (runs of workgroups with an incomplete last round) and
with rows of odd length, against the CPU oracle, bit for bit: every cell is
stepped exactly once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(g, o):
    assert np.array_equal(g.populations().view(np.uint8), o.fin.view(np.uint8))


@pytest.mark.parametrize("dim,st,sto,periodic", [
    ((131, 127, 109), "f32", 1, 0), ((131, 127, 109), "f32dev", 2, 2), ((99, 131, 277), "f16dev", 3, 0)])
def test_container_odd_rows_beyond_cache(nx, orc, dim, st, sto, periodic):
    g = nx.DenseLattice(dim, st, "f32", periodic=periodic)
    o = orc.DenseOracle(dim, sto, 1, periodic=periodic)
    assert 2 * 19 * g.populations().itemsize * np.prod(dim) > 256 << 20
    for lat in (g, o):
        lat.setup_cavity(0.05)
        lat.run(3, 1.7)
    _same(g, o)
    g.run_plain(2, 1.7)
    o.run(2, 1.7)
    _same(g, o)


def test_zouhe_beyond_cache(nx, orc):
    X, Y, Z = dim = (131, 127, 109)
    cls = np.full((Z, Y, X), 2, np.uint32)
    cls[:, [0, -1]] = cls[[0, -1]] = 0
    zh = np.zeros(cls.shape, np.uint32)
    zh[:, :, 0], zh[:, :, -1] = 1, 2
    zh[cls != 2] = 0
    g, o = nx.DenseLattice(dim, "f32", "f32"), orc.DenseOracle(dim, 1, 1)
    for lat in (g, o):
        lat.set_classes(cls.reshape(-1), zouhe=zh.reshape(-1))
        lat.run_zouhe(3, 1.4, [1.002, 0.998, 0, 0, 0, 0])
    _same(g, o)


def test_block_runs_beyond_cache(nx, orc):
    dim = (120, 120, 128)              # 3,600 blocks: the last round of 32 is incomplete
    act = np.ones(dim[::-1], np.uint8)
    act[40:56, 40:56, 40:56] = 0       # absent blocks inside
    grid = nx.BlockGrid(dim, act.reshape(-1))
    g, o = nx.BlockLattice(grid, "f32", "f32"), orc.BlockOracle(dim, act.reshape(-1), 1, 1)
    assert grid.n_blocks % 32 and grid.n_blocks * 512 * 38 * 4 > 256 << 20
    keep = o.active_slots()
    cls = np.where(keep, 2, 3).astype(np.uint32)
    for lat in (g, o):
        lat.set_classes(cls)
        lat.run(3, 1.7, force=(1e-5, 0.0, 0.0))
    k3 = keep.reshape(-1, 512)
    pg, po = (a.reshape(-1, 19, 512).transpose(1, 0, 2)[:, k3] for a in (g.populations(), o.fin))
    assert np.array_equal(pg, po)
