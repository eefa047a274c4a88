"""The staged convolution kernels at the edges of their tiles, against the FP64
oracle: rows of 4 to 64 voxels, fewer rows or planes than a tile, two tiles
along z, channel counts that end in a 16-channel slice, and infinities; and
runs of several rows, planes and chunks that end inside a column, a plane and a
sample.

Tolerance: as tests/test_gpu_conv.py -- every output sums at most 27 * 256
products in FP32, so it lies within 1e-5 of the sum of their magnitudes."""
import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu

SHAPES = [((1, 16, 16, 16), 80, 32), ((1, 32, 4, 16), 16, 48), ((1, 1, 1, 16), 32, 32), ((2, 64, 2, 8), 48, 16),
          ((1, 2, 1, 4), 48, 16), ((1, 4, 8, 4), 80, 32), ((1, 16, 4, 32), 48, 16), ((1, 2, 16, 32), 16, 48),
          ((3, 1, 1, 64), 16, 32), ((1, 16, 8, 64), 16, 16), ((2, 8, 2, 32), 112, 16)]
# Work of one workgroup: k_fwd_z16 3 planes of 8 (640 planes over 256 runs);
# k_bwd_wr 7 chunks = 3.5 rows of 64 voxels (5,120 chunks, 768 splits) and 7
# rows of 32 (1,280, 192 splits); k_bwd_wc the partials of a slice, each 3 of 11
# chunks (768 chunks, 70 splits), on rows of 8 and 4 one of 4, and one partial
# of 9 of 35 chunks (112 -> 16)
RUNS = [((5, 8, 64, 64), 16, 16), ((5, 8, 32, 32), 64, 32), ((6, 16, 16, 16), 32, 64), ((8, 16, 8, 8), 64, 32),
        ((8, 16, 8, 4), 48, 64), ((3, 16, 16, 16), 112, 16)]


def _bf(rng, shape, scale=1.0):
    bits = U.to_bf16_bits(rng.standard_normal(shape) * scale)
    return bits, U.from_bf16_bits(bits)


@pytest.mark.parametrize("shape,cin,cout", SHAPES + RUNS)
def test_rows_vs_oracle(nx, shape, cin, cout):
    from neon_amd import surrogate as S
    rng = np.random.default_rng(cin + cout)
    dev = nx.DeviceBuffer.from_array
    xb, x = _bf(rng, (*shape, cin))
    gb, g = _bf(rng, (*shape, cout))
    wb, w = _bf(rng, (cout, 27, cin), 0.2)
    V = int(np.prod(shape))
    y, dx = nx.DeviceBuffer(V * cout * 4), nx.DeviceBuffer(V * cin * 4)
    dw, db = nx.DeviceBuffer(cout * 27 * cin * 4), nx.DeviceBuffer(cout * 4)
    S.conv3d_fwd(dev(xb), dev(wb), None, y, shape, cin, cout, out_f32=True)
    S.conv3d_bwd_data(dev(gb), dev(wb), dx, shape, cin, cout, out_f32=True)
    S.conv3d_bwd_weight(dev(xb), dev(gb), dw, db, shape, cin, cout)
    ab = np.abs
    rw, rb = U.conv_bwd_weight(x, g, 3)
    bw, bb = U.conv_bwd_weight(ab(x), ab(g), 3)
    for got, ref, bound in ((y, U.conv_fwd(x, w, None, 3), U.conv_fwd(ab(x), ab(w), None, 3)),
                            (dx, U.conv_bwd_data(g, w, 3), U.conv_bwd_data(ab(g), ab(w), 3)), (dw, rw, bw), (db, rb, bb)):
        assert np.all(ab(got.download(np.float32).reshape(ref.shape) - ref) <= 1e-5 * bound + 1e-30)


@pytest.mark.parametrize("shape", [(1, 4, 4, 32), (1, 4, 4, 16), (1, 8, 4, 8), (1, 4, 4, 4)])
def test_weight_gradient_pairs_only_inside(nx, shape):
    """An infinite input voxel on the grid's faces reaches only the taps whose
    output voxel lies inside the grid; every other weight stays finite."""
    from neon_amd import surrogate as S
    n, D, H, W = shape
    x = np.ones((*shape, 16), np.float32)
    x[0, 0, H - 1, W // 2, 3] = np.inf
    g = np.ones((*shape, 16), np.float32)
    dw, db = nx.DeviceBuffer(16 * 27 * 16 * 4), nx.DeviceBuffer(16 * 4)
    dev = nx.DeviceBuffer.from_array
    S.conv3d_bwd_weight(dev(U.to_bf16_bits(x)), dev(U.to_bf16_bits(g)), dw, db, shape, 16, 16)
    got = dw.download(np.float32).reshape(16, 3, 3, 3, 16)
    for dz in range(3):
        for dy in range(3):
            for dx in range(3):
                z, y, v = 0 - (dz - 1), H - 1 - (dy - 1), W // 2 - (dx - 1)
                inside = 0 <= z < D and 0 <= y < H and 0 <= v < W
                assert np.all(np.isposinf(got[:, dz, dy, dx, 3]) if inside else np.isfinite(got[:, dz, dy, dx, 3]))
                assert np.all(np.isfinite(np.delete(got[:, dz, dy, dx], 3, axis=-1)))
