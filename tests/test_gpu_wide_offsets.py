"""The kernels with 64-bit offsets, which fields and levels of 4 GiB and more
take (the per-block step at 2-byte storage, the refinement path's stream at
every lattice and type), against those with 32-bit offsets on small grids, bit
for bit (nx_d3q19_set_wide_offsets)."""
import numpy as np
import pytest

from test_gpu_block import _raw, spheres

pytestmark = pytest.mark.gpu


@pytest.fixture
def wide(nx):
    from neon_amd import abi

    def set_wide(on):
        abi.check(abi.lib.nx_d3q19_set_wide_offsets(int(on)))
    yield set_wide
    set_wide(0)


@pytest.mark.parametrize("force", [(0.0, 0.0, 0.0), (1e-4, 0.0, -3e-5)])
def test_block_step(nx, wide, force):
    dim = (40, 24, 32)
    solid = spheres(dim, 12, 3, 7, seed=5)
    solid[:8, :8, :] = True
    grid = nx.BlockGrid(dim, (~solid).astype(np.uint8).reshape(-1), periodic=1)
    keep = np.unpackbits(grid.masks.view(np.uint8), bitorder="little").astype(bool)
    out = []
    for on in (0, 1):
        wide(on)
        lat = nx.BlockLattice(grid, "f16dev", "f32")
        lat.set_classes(np.where(keep, 2, 3).astype(np.uint32))
        lat.run(9, 1.7, force=force)
        out.append(_raw(lat.populations(), lat.storage))
    assert np.array_equal(*out)


@pytest.mark.parametrize("lattice", ["bgk19", "kbc27"])
@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("dim,shells", [((40, 36, 28), (0.0, -0.4, -1.0)), ((64, 48, 40), (0.0, -0.25, -0.6, -1.0))])
def test_refined_step(nx, wide, lattice, storage, dim, shells):
    from neon_amd import mgrid as mg
    out = []
    for on in (0, 1):
        wide(on)
        g = mg.MGrid(dim, list(mg.cavity_lambdas(dim, shells)), storage, lattice=lattice)
        g.setup_cavity(0.04)
        g.run(4, 1.3)
        out.append([g.fields(l, w) for l in range(g.depth) for w in (0, 1)])
    assert all(np.array_equal(a.view(np.uint8), b.view(np.uint8)) for a, b in zip(*out)) and np.any(out[0][0])
