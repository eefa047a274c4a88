"""The order in which a step deals workgroups to the XCDs -- slabs, as launched,
runs of workgroups with an incomplete last round -- on both sides of the field
sizes where it changes and with rows of odd length, against the CPU oracle, bit
for bit: every cell is stepped exactly once."""
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


@pytest.mark.parametrize("force", [(0.0, 0.0, 0.0), (1e-5, 0.0, 2e-6)])
@pytest.mark.parametrize("dim,st,sto", [((80, 72, 64), "f32", 1), ((45, 53, 40), "f32", 1), ((56, 72, 45), "f32dev", 2),
                                        ((83, 42, 43), "f64", 0), ((64, 50, 96), "f16dev", 3)])
def test_container_at_the_sizes_between(nx, orc, dim, st, sto, force):
    """Fields on both sides of the 48 MB up to which a step takes one slab per
    XCD (binary32: the interior-bitmap kernel either way), with obstacles."""
    X, Y, Z = dim
    rng = np.random.default_rng(X)
    cls = np.full((Z, Y, X), 2, np.uint32)
    cls[:, :, [0, -1]] = cls[:, [0, -1]] = cls[[0, -1]] = 0
    for _ in range(4):
        z, y, x = (int(rng.integers(2, n - 8)) for n in (Z, Y, X))
        cls[z:z + 5, y:y + 6, x:x + 7] = 0
    cm = 0 if st == "f64" else 1
    g, o = nx.DenseLattice(dim, st, "f64" if st == "f64" else "f32"), orc.DenseOracle(dim, sto, cm)
    for lat in (g, o):
        lat.set_classes(cls.reshape(-1))
        lat.run(5, 1.6, force=force)
    _same(g, o)


@pytest.mark.parametrize("dim,st,cm,mb", [((131, 127, 109), "f32", 1, 256), ((181, 151, 155), "f64", 0, 1200)])
def test_zouhe_large(nx, orc, dim, st, cm, mb):
    X, Y, Z = dim
    assert 38 * (8 if st == "f64" else 4) * X * Y * Z > mb << 20
    cls = np.full((Z, Y, X), 2, np.uint32)
    cls[:, [0, -1]] = cls[[0, -1]] = 0
    zh = np.zeros(cls.shape, np.uint32)
    zh[:, :, 0], zh[:, :, -1] = 1, 2
    zh[cls != 2] = 0
    g, o = nx.DenseLattice(dim, st, st), orc.DenseOracle(dim, cm, cm)
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
