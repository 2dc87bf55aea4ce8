"""Convolutions whose channel counts leave a partial K step in every filter tap, whose pixel count is no multiple of the K
step, or whose output is smaller than a tile: all of them can read their patch matrix in the GEMM's loader.  Called without
scratch and with less than the interim matrix needs (the reduction may then be split), where they do, and with what is asked for,
where they take the way that is expected to be faster; integers bit for bit against the oracle."""
import numpy as np
import pytest

from util import f, h, ints, rng

pytestmark = pytest.mark.gpu

# B, IH, IW, IC, OC, FH, FW, covered, sy, sx, dy, dx
CONV = [
    (2, 9, 7, 8, 8, 3, 3, True, 1, 1, 1, 1),       # a lone partial step per tap, fewer rows and columns than any tile
    (1, 12, 11, 72, 40, 3, 3, True, 1, 1, 1, 1),   # a whole step and a piece of one
    (3, 15, 15, 96, 136, 3, 3, True, 2, 2, 1, 1),  # strided: the gradient of x by classes
    (2, 14, 13, 56, 64, 1, 1, True, 1, 1, 1, 1),   # one tap
    (2, 13, 17, 24, 160, 5, 5, False, 1, 1, 1, 1),
    (4, 21, 10, 40, 16, 3, 3, True, 1, 1, 2, 2),
]
# B, IH, IW, IC, OC, FH, FW, covered, sy, sx
DECONV = [
    (2, 7, 7, 96, 40, 4, 4, False, 2, 2),
    (1, 5, 6, 8, 8, 3, 3, False, 2, 2),            # classes of a few pixels
    (3, 6, 9, 40, 72, 2, 2, False, 2, 2),
    (2, 10, 10, 24, 136, 3, 3, True, 1, 1),
]


def _call(lib, name, dt, bufs, shape, filt, geo, out, scratch_bytes):
    from deep8_amd.capi import DeviceArray, check
    a, b, c = bufs
    ws = DeviceArray((max(scratch_bytes, 16),), np.uint8)
    check(getattr(lib, name)(dt, a.ptr, *shape, b.ptr, *filt, c.ptr, *geo, ws.ptr if scratch_bytes else None, scratch_bytes, None))
    return f(out.numpy())


@pytest.mark.parametrize("op,cfg", [("conv2d", c) for c in CONV] + [("deconv2d", c) for c in DECONV])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_partial_steps_without_interim_matrix(oracle_port, op, cfg, dtype):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray
    lib = capi.init()
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = getattr(ops, op + "_geometry")(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]))
    hi = 3 if dtype == np.float16 else 10
    c = (lambda v: h(v)) if dtype == np.float16 else (lambda v: v)
    x, w, gz = ints(r, (B, IH, IW, IC), hi), ints(r, (OC, FH, FW, IC), hi), ints(r, (B, OH, OW, OC), hi)
    if dtype == np.float16:  # thinned, so that every sum stays a whole number that half can hold
        x, w, gz = x * (r.random(x.shape) < 0.3), w * (r.random(w.shape) < 0.3), gz * (r.random(gz.shape) < 0.3)
    port = oracle_port
    want = [getattr(port, op)(x, w, *geo), getattr(port, op + "_grad_x")(x, w, gz, *geo), getattr(port, op + "_grad_y")(x, w, gz, *geo)]
    assert dtype == np.float32 or max(np.abs(t).max() for t in want) < 2048
    dt = capi.dtype_id(np.dtype(dtype))
    shape, filt, g = (B, IH, IW, IC), (OC, FH, FW), (int(geo[0]),) + tuple(geo[1:])
    for which, name in enumerate(("d8_" + op, "d8_%s_grad_x_overwrite" % op, "d8_%s_grad_y_overwrite" % op)):
        nan = DeviceArray.from_numpy(np.full(want[which].shape, np.nan, dtype))
        bufs = [DeviceArray.from_numpy(c(x)), DeviceArray.from_numpy(c(w)), DeviceArray.from_numpy(c(gz))]
        bufs[(2, 0, 1)[which]] = nan
        asked = getattr(lib, "d8_%s_scratch_bytes" % op)(dt, which, *shape, *filt, *g)
        interim = (B * OH * OW * IC if op == "conv2d" else B * IH * IW * OC) * FH * FW * np.dtype(dtype).itemsize
        for scratch in (0, interim - 16, asked):
            before = lib.d8_conv_route_calls(1)
            got = _call(lib, name, dt, bufs, shape, filt, g, nan, scratch)
            assert np.array_equal(got, want[which]), (which, scratch)
            assert scratch == asked or lib.d8_conv_route_calls(1) == before + 1


# op, which, element type, layer, the way it has to go with all the scratch it asks for (0 interim matrix, 1 loader, 2 LDS): both
# sides were measured, in us, on the matrix / in the loader / from LDS
ROUTES = [
    ("conv2d", 0, np.float32, (3, 15, 15, 48, 140, 3, 3, True, 2, 2, 1, 1), 0),      # 10 / 46
    ("conv2d", 0, np.float32, (2, 46, 46, 8, 128, 3, 3, True, 1, 1, 1, 1), 0),       # a quarter of every K step is not padding
    ("conv2d", 0, np.float16, (3, 15, 15, 96, 136, 3, 3, True, 2, 2, 1, 1), 1),
    ("conv2d", 1, np.float32, (5, 10, 7, 152, 512, 5, 5, True, 2, 2, 1, 1), 0),      # 23 / 275
    ("conv2d", 1, np.float32, (10, 20, 20, 32, 96, 3, 3, True, 2, 2, 1, 1), 1),
    ("conv2d", 1, np.float32, (14, 8, 8, 224, 24, 1, 1, False, 2, 2, 1, 1), 0),      # 9 / 14: three of four pixels have no tap
    ("conv2d", 2, np.float32, (29, 13, 13, 40, 128, 3, 3, True, 2, 2, 1, 1), 0),     # 10 / 35
    ("conv2d", 2, np.float16, (9, 30, 30, 96, 160, 3, 3, True, 2, 2, 1, 1), 1),
    ("conv2d", 2, np.float16, (6, 137, 137, 3, 142, 3, 3, True, 1, 1, 1, 1), 0),     # (17 images) 73 / - / 430
    ("conv2d", 2, np.float16, (4, 56, 56, 3, 64, 7, 7, True, 2, 2, 1, 1), 2),
    ("conv2d", 0, np.float32, (64, 28, 28, 1, 32, 5, 5, True, 1, 1, 1, 1), 2),       # 18 / - / 8
    ("deconv2d", 0, np.float32, (1, 7, 7, 128, 448, 3, 3, False, 1, 1), 0),          # 14 / 74
    ("deconv2d", 0, np.float16, (6, 12, 12, 96, 40, 4, 4, False, 2, 2), 1),
    ("deconv2d", 1, np.float32, (6, 5, 5, 160, 8, 4, 4, False, 2, 2), 0),            # 7 / 37
    ("deconv2d", 2, np.float16, (6, 11, 11, 160, 32, 4, 4, False, 2, 2), 0),         # 12 / 19
]


@pytest.mark.parametrize("op,which,dtype,cfg,route", ROUTES)
def test_the_way_a_layer_goes(op, which, dtype, cfg, route):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = (int(cfg[7]),) + cfg[8:]
    OH, OW, _, _ = getattr(ops, op + "_geometry")(IH, IW, FH, FW, *cfg[7:])
    dt, shape, filt = capi.dtype_id(np.dtype(dtype)), (B, IH, IW, IC), (OC, FH, FW)
    x, w, z = (DeviceArray(s, dtype, zero=True) for s in (shape, (OC, FH, FW, IC), (B, OH, OW, OC)))
    name = ("d8_" + op, "d8_%s_grad_x_overwrite" % op, "d8_%s_grad_y_overwrite" % op)[which]
    asked = getattr(lib, "d8_%s_scratch_bytes" % op)(dt, which, *shape, *filt, *geo)
    ws = DeviceArray((max(asked, 16),), np.uint8)
    before = [lib.d8_conv_route_calls(k) for k in range(3)]
    check(getattr(lib, name)(dt, x.ptr, *shape, w.ptr, *filt, z.ptr, *geo, ws.ptr, asked, None))
    assert [lib.d8_conv_route_calls(k) - before[k] for k in range(3)] == [int(k == route) for k in range(3)]


def test_scratch_that_starts_anywhere_is_no_room_for_the_matrix(oracle_port):
    """a layer that goes over the matrix with the scratch it asks for reads its patches in the loader when that is not aligned"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(5)
    x, w = ints(r, (3, 15, 15, 48), 4), ints(r, (140, 3, 3, 48), 4)
    want = oracle_port.conv2d(x, w, True, 2, 2, 1, 1)
    args = (3, 15, 15, 48), (140, 3, 3), (1, 2, 2, 1, 1)
    asked = lib.d8_conv2d_scratch_bytes(capi.FLOAT32, 0, *args[0], *args[1], *args[2])
    dx, dw, ws = DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), DeviceArray((asked + 16,), np.uint8)
    for shift, route in ((0, 0), (4, 1)):
        dz = DeviceArray.from_numpy(np.full(want.shape, np.nan, np.float32))
        before = lib.d8_conv_route_calls(route)
        check(lib.d8_conv2d(capi.FLOAT32, dx.ptr, *args[0], dw.ptr, *args[1], dz.ptr, *args[2], ws.ptr + shift, asked, None))
        assert lib.d8_conv_route_calls(route) == before + 1 and np.array_equal(dz.numpy(), want)


def test_pixels_past_the_last_of_a_large_image():
    """one output pixel on an image of 77 MB: the 63 pixels that fill the K step up lie up to 4.9 GB past the image, whose other
    elements (NaN) they must not meet"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    size, IC, OC, F = 2200, 8, 64, 3
    geo = (0, size, size, 1, 1)
    x = np.full((1, size, size, IC), np.nan, np.float16)
    r = rng(5)
    x[0, :F, :F] = ints(r, (F, F, IC), 5)
    gz = ints(r, (1, 1, 1, OC), 5)
    want = gz.reshape(OC, 1, 1, 1) * f(x[:, :F, :F])
    shape, filt = (1, size, size, IC), (OC, F, F)
    need = lib.d8_conv2d_scratch_bytes(capi.FLOAT16, 2, *shape, *filt, *geo)
    dx, dg, out = DeviceArray.from_numpy(x), DeviceArray.from_numpy(h(gz)), DeviceArray.from_numpy(np.full(want.shape, np.nan, np.float16))
    ws = DeviceArray((need,), np.uint8)
    check(lib.d8_conv2d_grad_y_overwrite(capi.FLOAT16, dx.ptr, *shape, out.ptr, *filt, dg.ptr, *geo, ws.ptr, need, None))
    assert np.array_equal(f(out.numpy()), want)
