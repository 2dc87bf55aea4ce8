"""Convolutions, both gradients from one call, on layers whose two products are tiled and cut as they would be alone and
share a launch: classes of output pixels (strides above 1), last K steps that are cut short, gradients of x in pieces.  Channels
narrower and wider than a tile, classes that no tap reaches, one-pixel classes, dilation, every combination of written and added
gradients, scratch for no pieces.  Integers, against the oracle, bit for bit; reals, bit for bit what two launches leave; and which
calls share one is counted."""
import numpy as np
import pytest

from util import f, ints, nrm, rng

pytestmark = pytest.mark.gpu

# B, IH, IW, IC, OC, FH, FW, covered, sy, sx, dy, dx
LAYERS = [
    (4, 17, 15, 64, 64, 3, 3, True, 2, 2, 1, 1),      # 128 x 64 tiles, whole K steps
    (3, 19, 21, 96, 160, 3, 3, True, 2, 2, 1, 1),     # K steps cut short
    (8, 16, 16, 136, 72, 3, 3, False, 2, 2, 1, 1),    # 128 x 128 tiles, columns past a tile
    (16, 18, 18, 64, 64, 1, 1, True, 2, 2, 1, 1),     # three classes that no tap reaches
    (12, 20, 20, 128, 128, 2, 2, False, 3, 3, 1, 1),  # five of nine
    (6, 16, 18, 64, 128, 3, 3, True, 2, 1, 1, 2),     # one stride, dilation along the other axis
    (4, 17, 17, 72, 64, 5, 5, True, 2, 2, 1, 1),
    (32, 3, 4, 64, 64, 3, 3, True, 2, 2, 1, 1),       # classes of one row and column
    (2, 40, 40, 256, 192, 3, 3, True, 2, 2, 1, 1),    # filter gradient on 128 x 128 tiles
    (3, 19, 21, 96, 160, 3, 3, True, 1, 1, 1, 1),     # stride 1, K steps cut short
    (6, 13, 13, 56, 72, 3, 3, False, 1, 1, 2, 1),     # 64 x 64 tiles of few columns
    (8, 11, 11, 256, 128, 5, 5, True, 1, 1, 1, 1),    # gradient of x in pieces
    (16, 28, 28, 136, 88, 3, 3, True, 1, 1, 1, 1),    # 128 x 128 tiles, columns past a tile
]
# (fp32: 128 x 32 tiles; in half the first would run whole in company, in pieces alone)
NARROW = [(16, 14, 14, 32, 64, 5, 5, True, 1, 1, 1, 1), (7, 28, 28, 32, 40, 3, 3, True, 2, 2, 1, 1)]
# fp32, on either side of the limit of workgroups, with and without pieces
CROWDED = [
    (64, 14, 14, 32, 64, 5, 5, True, 1, 1, 1, 1),     # 128 x 32 tiles beside 64 x 128: any number
    (64, 14, 14, 28, 40, 3, 3, True, 1, 1, 1, 1),
    (12, 28, 28, 136, 168, 3, 3, True, 1, 1, 1, 1),   # filter gradient on 128 x 128 tiles: two a compute unit
    (24, 28, 28, 136, 88, 3, 3, True, 1, 1, 1, 1),
    (6, 67, 67, 64, 64, 3, 3, True, 1, 1, 1, 1),      # 128 x 64 tiles: two a compute unit
    (8, 40, 40, 136, 136, 3, 3, True, 1, 1, 1, 1),    # 128 x 128 tiles in both: never
]
# With the scratch that is asked for these run apart: their patch matrix is expected to be faster, or (fp32) pieces make more
# workgroups than a compute unit holds two of.
APART = [(LAYERS[i], np.float32) for i in (1, 2, 4, 7, 9, 10, 11)] + [(LAYERS[5], np.float16)] + [(CROWDED[i], np.float32) for i in (2, 3, 4, 5)]
# ... and these without scratch: shared whole by the older rule, or never
APART_WHOLE = [(NARROW[0], np.float32), (CROWDED[0], np.float32), (CROWDED[5], np.float32)]

# B, IH, IW, IC, OC, FH, FW, covered, sy, sx
TRANSPOSED = [
    (4, 14, 13, 64, 72, 4, 4, False, 2, 2),
    (2, 9, 11, 136, 40, 3, 3, True, 2, 2),            # too small for tiles
    (18, 6, 6, 72, 16, 5, 5, False, 2, 2),
    (6, 16, 16, 64, 200, 3, 3, False, 1, 1),
    (8, 20, 20, 128, 88, 2, 2, False, 2, 2),
    (4, 12, 12, 136, 136, 3, 3, False, 2, 2),
]
APART_TRANSPOSED = [(TRANSPOSED[0], np.float16), (TRANSPOSED[1], np.float32), (TRANSPOSED[1], np.float16)]
APART_TRANSPOSED_WHOLE = APART_TRANSPOSED[1:]


def _layer(name, cfg, dtype, x, w, gz):
    """call(gx0, gw0, overwrite, scratch bytes) -> both gradients and how many launches were shared; the scratch asked for"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt, (B, IH, IW, IC, OC, FH, FW), geo = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32, cfg[:7], tuple(int(v) for v in cfg[7:])
    dx, dw, dgz = (DeviceArray.from_numpy(np.asarray(t, dtype)) for t in (x, w, gz))

    def call(gx0, gw0, overwrite, nb):
        gx, gw, ws = DeviceArray.from_numpy(np.asarray(gx0, dtype)), DeviceArray.from_numpy(np.asarray(gw0, dtype)), DeviceArray((max(nb, 16),), np.uint8)
        before = lib.d8_conv_grad_kept_pair_launches()
        check(getattr(lib, f"d8_{name}_grad_xy")(dt, dx.ptr, gx.ptr, B, IH, IW, IC, dw.ptr, gw.ptr, OC, FH, FW, dgz.ptr, *geo, overwrite,
                                                 ws.ptr if nb else None, nb, None))
        return gx.numpy(), gw.numpy(), lib.d8_conv_grad_kept_pair_launches() - before

    return call, getattr(lib, f"d8_{name}_scratch_bytes")(dt, 3, B, IH, IW, IC, OC, FH, FW, *geo)


def _shares(cfg, dtype, nb, apart, apart_whole):
    return int((cfg, dtype) not in (apart if nb else apart_whole))


@pytest.mark.parametrize("cfg", LAYERS)
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_integers_against_the_oracle(oracle_port, cfg, dtype):
    from deep8_amd import ops
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]))
    x, w, gz = ints(r, (B, IH, IW, IC), 2), ints(r, (OC, FH, FW, IC), 2), ints(r, (B, OH, OW, OC), 2)
    gz = gz * (r.random(gz.shape) < min(1.0, 400.0 / (B * OH * OW)))  # thinned: sums that half holds
    gx0, gw0 = ints(r, x.shape, 2), ints(r, w.shape, 2)
    want_x, want_w = oracle_port.conv2d_grad_x(x, w, gz, *geo), oracle_port.conv2d_grad_y(x, w, gz, *geo)
    assert max(np.abs(want_x).max(), np.abs(want_w).max()) < 2000
    call, asked = _layer("conv2d", cfg, dtype, x, w, gz)
    for nb in (0, asked):
        for overwrite in (3, 2, 1, 0):
            gx, gw, shared = call(gx0, gw0, overwrite, nb)
            assert shared == _shares(cfg, dtype, nb, APART, APART_WHOLE), nb
            assert np.array_equal(f(gx), want_x + (0 if overwrite & 1 else gx0)), (nb, overwrite)
            assert np.array_equal(f(gw), want_w + (0 if overwrite & 2 else gw0)), (nb, overwrite)


@pytest.mark.parametrize("cfg,dtype", [(c, t) for c in LAYERS for t in (np.float32, np.float16)] + [(c, np.float32) for c in NARROW + CROWDED])
def test_one_launch_leaves_what_two_leave(cfg, dtype, monkeypatch):
    from deep8_amd import ops
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]) + 1)
    x, w, gz = (nrm(r, s) for s in ((B, IH, IW, IC), (OC, FH, FW, IC), (B, OH, OW, OC)))
    call, asked = _layer("conv2d", cfg, dtype, x, w, gz)
    for nb in (0, asked):
        monkeypatch.delenv("D8_CONV_GRADS_APART", raising=False)
        one = call(np.full(x.shape, np.nan), np.full(w.shape, np.nan), 3, nb)
        monkeypatch.setenv("D8_CONV_GRADS_APART", "1")
        two = call(np.full(x.shape, np.nan), np.full(w.shape, np.nan), 3, nb)
        assert (one[2], two[2]) == (_shares(cfg, dtype, nb, APART, APART_WHOLE), 0), nb
        assert all(np.array_equal(a.view(np.uint8), b.view(np.uint8)) for a, b in zip(one[:2], two[:2])), nb


@pytest.mark.parametrize("cfg", TRANSPOSED)
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_transposed_convolutions(oracle_port, cfg, dtype, monkeypatch):
    from deep8_amd import ops
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = ops.deconv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]) + 2)
    for whole in (True, False):
        if whole:
            x, w, gz = ints(r, (B, IH, IW, IC), 2), ints(r, (OC, FH, FW, IC), 2), ints(r, (B, OH, OW, OC), 2)
            x = x * (r.random(x.shape) < min(1.0, 400.0 / (B * IH * IW)))  # thinned: sums that half holds
            gz = gz * (r.random(gz.shape) < 0.3)
        else:
            x, w, gz = nrm(r, (B, IH, IW, IC)), nrm(r, (OC, FH, FW, IC)), nrm(r, (B, OH, OW, OC))
        gx0, gw0 = ints(r, x.shape, 2), ints(r, w.shape, 2)
        call, asked = _layer("deconv2d", cfg, dtype, x, w, gz)
        for nb in (0, asked):
            for overwrite in (3, 0):
                monkeypatch.delenv("D8_CONV_GRADS_APART", raising=False)
                one = call(gx0, gw0, overwrite, nb)
                monkeypatch.setenv("D8_CONV_GRADS_APART", "1")
                two = call(gx0, gw0, overwrite, nb)
                assert (one[2], two[2]) == (_shares(cfg, dtype, nb, APART_TRANSPOSED, APART_TRANSPOSED_WHOLE), 0), nb
                assert all(np.array_equal(a.view(np.uint8), b.view(np.uint8)) for a, b in zip(one[:2], two[:2])), nb
                if whole:
                    want_x, want_w = oracle_port.deconv2d_grad_x(x, w, gz, *geo), oracle_port.deconv2d_grad_y(x, w, gz, *geo)
                    assert max(np.abs(want_x).max(), np.abs(want_w).max()) < 2000
                    assert np.array_equal(f(one[0]), want_x + (0 if overwrite else gx0))
                    assert np.array_equal(f(one[1]), want_w + (0 if overwrite else gw0))
