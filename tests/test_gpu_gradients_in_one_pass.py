"""Both gradients of half layers of few tiles: what shares a launch with a longer product is not cut into pieces for it, so nothing is
written to the scratch and there is no second pass; and into no more than its tiles' times ask for.  Integers, bit for bit."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


def _untouched(ws):
    return np.array_equal(ws.numpy(), np.full(ws.numpy().shape, 0xff, np.uint8))


@pytest.mark.parametrize("xb,R,I,O", [(4, 320, 128, 1408), (1, 576, 128, 1216), (1, 1792, 256, 1088)])
def test_matmul(xb, R, I, O):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    sparse = lambda *s: ints(r, s, 2) * (r.random(s) < 0.25)
    x, y, dz = sparse(xb, R, I), sparse(xb, I, O), sparse(xb, R, O)
    wx, wy = np.matmul(dz, y.transpose(0, 2, 1)), np.matmul(x.transpose(0, 2, 1), dz)
    assert max(np.abs(wx).max(), np.abs(wy).max()) < 2048
    nb = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 3, xb, R, I, xb, I, O)
    dx, dy, dd = (DeviceArray.from_numpy(t.astype(np.float16)) for t in (x, y, dz))
    gx, gy = DeviceArray.from_numpy(np.full(x.shape, np.nan, np.float16)), DeviceArray.from_numpy(np.full(y.shape, np.nan, np.float16))
    ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
    check(lib.d8_matmul_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, xb, R, I, dy.ptr, gy.ptr, xb, I, O, dd.ptr, 3, ws.ptr, nb, None))
    assert np.array_equal(gx.numpy(), wx.astype(np.float16)) and np.array_equal(gy.numpy(), wy.astype(np.float16))
    assert _untouched(ws)


@pytest.mark.parametrize("R,I,O,pieces", [(4560, 1216, 64, 12), (4056, 1416, 64, 11)])
def test_pieces_of_the_second_gradient(R, I, O, pieces):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R)
    sparse = lambda *s: ints(r, s, 2) * (r.random(s) < 0.25)
    x, y, dz = sparse(R, I), sparse(I, O), sparse(R, O)
    wx, wy = dz @ y.T, x.T @ dz
    assert max(np.abs(wx).max(), np.abs(wy).max()) < 2048
    nb = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 3, 1, R, I, 1, I, O)
    dx, dy, dd = (DeviceArray.from_numpy(t.astype(np.float16)) for t in (x, y, dz))
    gx, gy = DeviceArray.from_numpy(np.full(x.shape, np.nan, np.float16)), DeviceArray.from_numpy(np.full(y.shape, np.nan, np.float16))
    ws = DeviceArray.from_numpy(np.full(nb // 4, np.nan, np.float32))
    check(lib.d8_matmul_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, 1, R, I, dy.ptr, gy.ptr, 1, I, O, dd.ptr, 3, ws.ptr, nb, None))
    assert np.array_equal(gx.numpy(), wx.astype(np.float16)) and np.array_equal(gy.numpy(), wy.astype(np.float16))
    written = ~np.isnan(ws.numpy())
    assert written[:pieces * I * O].all() and not written[pieces * I * O:].any()


def test_conv2d(oracle_port):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    image, filt, geo = (2, 19, 19, 64), (128, 3, 3), (1, 1, 1, 1, 1)
    r = rng(19)
    sparse = lambda *s: ints(r, s, 2) * (r.random(s) < 0.25)
    x, w, dz = sparse(*image), sparse(*filt, 64), sparse(2, 19, 19, 128)
    nb = lib.d8_conv2d_scratch_bytes(capi.FLOAT16, 3, *image, *filt, *geo)
    dx, dw, dd = (DeviceArray.from_numpy(t.astype(np.float16)) for t in (x, w, dz))
    gx, gw = DeviceArray.from_numpy(np.full(x.shape, np.nan, np.float16)), DeviceArray.from_numpy(np.full(w.shape, np.nan, np.float16))
    ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
    check(lib.d8_conv2d_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, *image, dw.ptr, gw.ptr, *filt, dd.ptr, *geo, 3, ws.ptr, nb, None))
    wx, ww = oracle_port.conv2d_grad_x(x, w, dz, *geo), oracle_port.conv2d_grad_y(x, w, dz, *geo)
    assert np.array_equal(gx.numpy(), wx.astype(np.float16)) and np.array_equal(gw.numpy(), ww.astype(np.float16))
    assert _untouched(ws)
