"""The convolutions' sums keep their order: every output equals, bit for bit,
that of the first kernels of this library (one staged tile, or one tap, per
workgroup), whose digests tests/golden/conv_sums.json holds.  A network
multiplies one changed bf16 rounding some 20 times a layer, so a kernel that
adds in another order changes what a training run gives.

The shapes take every kernel through several rows, planes, columns or chunks of
one workgroup, across samples, and through its last partial run; thin grids,
rows of 1 to 128 voxels, channel counts that end in half a slice.
`python tests/test_gpu_conv_order.py FILE` writes the digests of the library
that is there."""
import hashlib
import json
import pathlib

import numpy as np
import pytest

from oracle import unet_oracle as U

GOLDEN = pathlib.Path(__file__).parent / "golden" / "conv_sums.json"
SHAPES = [((5, 8, 64, 64), 16, 16, 3), ((3, 16, 32, 32), 64, 64, 3), ((2, 8, 16, 64), 48, 32, 3), ((3, 8, 8, 32), 112, 48, 3),
          ((1, 4, 4, 64), 16, 48, 3), ((2, 4, 8, 128), 32, 16, 3), ((2, 2, 8, 64), 16, 32, 3), ((1, 8, 2, 32), 48, 16, 3),
          ((6, 16, 16, 16), 32, 64, 3), ((2, 4, 8, 16), 80, 48, 3), ((2, 4, 4, 16), 256, 64, 3), ((1, 8, 16, 16), 144, 32, 3),
          ((8, 16, 8, 8), 64, 32, 3), ((2, 4, 4, 8), 176, 16, 3), ((3, 8, 4, 8), 16, 64, 3),
          ((8, 16, 8, 4), 48, 64, 3), ((2, 4, 4, 4), 256, 32, 3), ((2, 2, 16, 4), 64, 16, 3),
          ((3, 8, 8, 2), 48, 32, 3), ((2, 4, 4, 1), 16, 16, 3), ((3, 1, 1, 64), 32, 16, 3),
          ((3, 16, 16, 16), 112, 16, 3), ((8, 8, 8, 8), 16, 112, 3), ((16, 8, 8, 4), 112, 16, 3),
          ((3, 16, 16, 16), 48, 16, 1), ((2, 8, 8, 8), 32, 80, 1), ((1, 1, 2, 4), 64, 64, 1)]
NETS = [(32, (16, 32, 64), 3), (64, (16, 32), 2)]


def _digest(a):
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()[:16]


def conv_digests(nx, shape, cin, cout, ks):
    from neon_amd import surrogate as S
    rng = np.random.default_rng(cin + 7 * cout + ks)
    V, T = int(np.prod(shape)), ks ** 3
    up = lambda n, s: nx.DeviceBuffer.from_array(U.to_bf16_bits(rng.standard_normal(n) * s))
    x, g, w = up(V * cin, 1.0), up(V * cout, 1e-3), up(cout * T * cin, 0.2)
    b = nx.DeviceBuffer.from_array(rng.standard_normal(cout).astype(np.float32))
    y, y32, dx = nx.DeviceBuffer(V * cout * 2), nx.DeviceBuffer(V * cout * 4), nx.DeviceBuffer(V * cin * 2)
    dw, db = nx.DeviceBuffer(cout * T * cin * 4), nx.DeviceBuffer(cout * 4)
    S.conv3d_fwd(x, w, b, y, shape, cin, cout, ks, relu=True)
    S.conv3d_fwd(x, w, None, y32, shape, cin, cout, ks, out_f32=True)
    S.conv3d_bwd_data(g, w, dx, shape, cin, cout, ks)
    S.conv3d_bwd_weight(x, g, dw, db, shape, cin, cout, ks)
    return {k: _digest(v.download(np.uint8)) for k, v in dict(y=y, y32=y32, dx=dx, dw=dw, db=db).items()}


def net_digests(nx, size, widths, batch):
    """Loss, gradients and weights after three training steps."""
    from neon_amd import surrogate as S
    rng = np.random.default_rng(size)
    net, V = S.UNet(size, len(widths), list(widths), batch, seed=5), batch * size ** 3
    x, t, w = (nx.DeviceBuffer.from_array(rng.random(V * c, np.float32) * s) for c, s in ((3, 1.0), (4, 1.0), (1, 1.0 / V)))
    for _ in range(3):
        loss = net.train_step(x, t, w, batch, 5e-4, want_loss=True)
    return {"loss": float(loss).hex(), "grads": _digest(net.grads()), "params": _digest(net.params())}


def every(nx):
    return {**{f"{s} {ci} {co} {ks}": conv_digests(nx, s, ci, co, ks) for s, ci, co, ks in SHAPES},
            **{f"net {n[0]} {n[1]} {n[2]}": net_digests(nx, *n) for n in NETS}}


@pytest.mark.gpu
@pytest.mark.parametrize("shape,cin,cout,ks", SHAPES)
def test_conv_sums(nx, shape, cin, cout, ks):
    assert conv_digests(nx, shape, cin, cout, ks) == json.loads(GOLDEN.read_text())[f"{shape} {cin} {cout} {ks}"]


@pytest.mark.gpu
@pytest.mark.parametrize("size,widths,batch", NETS)
def test_training_steps(nx, size, widths, batch):
    assert net_digests(nx, size, widths, batch) == json.loads(GOLDEN.read_text())[f"net {size} {widths} {batch}"]


if __name__ == "__main__":
    import sys
    import neon_amd
    neon_amd.init()
    pathlib.Path(sys.argv[1]).write_text(json.dumps(every(neon_amd), indent=0) + "\n")
