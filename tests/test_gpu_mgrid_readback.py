"""Read-back of a refined level (nx_mgrid_fields): only active voxels of the
caller's array are written, also where a level has partial blocks, inactive
interiors and more values than one read-back chunk, or so few that it is copied
without the chunks."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lattice,storage", [((40, 36, 28), "bgk19", "f32"), ((64, 48, 72), "kbc27", "f64"),
                                                 ((17, 13, 9), "bgk19", "f64"), ((17, 13, 9), "bgk19", "f32"),
                                                 ((24, 24, 24), "kbc27", "f32")])
def test_inactive_voxels_keep_the_callers_values(nx, dim, lattice, storage):
    from neon_amd import mgrid as mg
    g = mg.MGrid(dim, list(mg.cavity_lambdas(dim, (0.0, -0.4, -1.0))), storage, lattice=lattice)
    g.setup_cavity(0.04)
    g.run(3, 1.2)
    for lvl in range(g.depth):
        for which in (0, 1):
            plain = g.fields(lvl, which)
            act = np.tile((g.state(lvl) & 1).astype(bool), g.Q)
            assert not plain[~act].any() and np.isfinite(plain).all() and plain[act].any()
            keep = np.full(plain.size, 7.0, plain.dtype)
            nx.abi.check(nx.abi.lib.nx_mgrid_fields(g.h, lvl, which, keep.ctypes.data_as(C.c_void_p)))
            assert np.array_equal(keep, np.where(act, plain, 7.0))
