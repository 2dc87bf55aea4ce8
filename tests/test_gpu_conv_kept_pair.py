"""Convolutions, both gradients from one call, on layers whose two products are tiled and cut as they would be alone and
share a launch: classes of output pixels (strides above 1), last K steps that are cut short, gradients of x in pieces.  Channels
narrower and wider than a tile, classes that no tap reaches, one-pixel classes, dilation, every combination of written and added
gradients, scratch for no pieces.  Integers, against the oracle, bit for bit; reals, bit for bit what two launches leave."""
import numpy as np
import pytest

from util import f, h, ints, nrm, rng

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


@pytest.mark.parametrize("cfg", LAYERS)
def test_integers_against_the_oracle(oracle_port, cfg):
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
    for ox, ow in ((True, True), (False, True), (True, False), (False, False)):
        gx, gw = ops.conv2d_grad_xy(h(x), h(w), h(gz), *geo, h(gx0), h(gw0), ox, ow)
        assert np.array_equal(f(gx), want_x + (0 if ox else gx0)), (ox, ow)
        assert np.array_equal(f(gw), want_w + (0 if ow else gw0)), (ox, ow)


# (fp32: 128 x 32 tiles; in half the first would run whole in company, in pieces alone)
NARROW = [(16, 14, 14, 32, 64, 5, 5, True, 1, 1, 1, 1), (7, 28, 28, 32, 40, 3, 3, True, 2, 2, 1, 1)]


@pytest.mark.parametrize("cfg,dtype", [(c, t) for c in LAYERS for t in (np.float32, np.float16)] + [(c, np.float32) for c in NARROW])
def test_one_launch_leaves_what_two_leave(cfg, dtype, monkeypatch):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r, dt = rng(sum(cfg[:7]) + 1), capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    x, w, gz = (DeviceArray.from_numpy(nrm(r, s).astype(dtype)) for s in ((B, IH, IW, IC), (OC, FH, FW, IC), (B, OH, OW, OC)))
    asked = lib.d8_conv2d_scratch_bytes(dt, 3, B, IH, IW, IC, OC, FH, FW, *(int(v) for v in geo))
    for nb in (0, asked):
        got = []
        for apart in (False, True):
            if apart:
                monkeypatch.setenv("D8_CONV_GRADS_APART", "1")
            else:
                monkeypatch.delenv("D8_CONV_GRADS_APART", raising=False)
            gx, gw = (DeviceArray.from_numpy(np.full(s, np.nan, dtype)) for s in ((B, IH, IW, IC), (OC, FH, FW, IC)))
            ws = DeviceArray((max(nb, 16),), np.uint8)
            check(lib.d8_conv2d_grad_xy(dt, x.ptr, gx.ptr, B, IH, IW, IC, w.ptr, gw.ptr, OC, FH, FW, gz.ptr,
                                        *(int(v) for v in geo), 3, ws.ptr if nb else None, nb, None))
            got.append((gx.numpy().view(np.uint8), gw.numpy().view(np.uint8)))
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]), nb


# B, IH, IW, IC, OC, FH, FW, covered, sy, sx
TRANSPOSED = [
    (4, 14, 13, 64, 72, 4, 4, False, 2, 2),
    (2, 9, 11, 136, 40, 3, 3, True, 2, 2),
    (18, 6, 6, 72, 16, 5, 5, False, 2, 2),
    (6, 16, 16, 64, 200, 3, 3, False, 1, 1),
    (8, 20, 20, 128, 88, 2, 2, False, 2, 2),
]


@pytest.mark.parametrize("cfg", TRANSPOSED)
def test_transposed_convolutions(oracle_port, cfg, monkeypatch):
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
        for ox, ow in ((True, True), (False, False)):
            monkeypatch.delenv("D8_CONV_GRADS_APART", raising=False)
            one = ops.deconv2d_grad_xy(h(x), h(w), h(gz), *geo, h(gx0), h(gw0), ox, ow)
            monkeypatch.setenv("D8_CONV_GRADS_APART", "1")
            two = ops.deconv2d_grad_xy(h(x), h(w), h(gz), *geo, h(gx0), h(gw0), ox, ow)
            assert all(np.array_equal(a.view(np.uint16), b.view(np.uint16)) for a, b in zip(one, two))
            if whole:
                want_x, want_w = oracle_port.deconv2d_grad_x(x, w, gz, *geo), oracle_port.deconv2d_grad_y(x, w, gz, *geo)
                assert max(np.abs(want_x).max(), np.abs(want_w).max()) < 2000
                assert np.array_equal(f(one[0]), want_x + (0 if ox else gx0))
                assert np.array_equal(f(one[1]), want_w + (0 if ow else gw0))
