"""Gradients that run longer in one launch than in two (a few workgroups more than the chip holds at once, of products that fill
their own rounds): they run apart, and those beside them share.  Integers, bit for bit."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,R,I,O,shared", [(np.float32, 4352, 448, 832, 0), (np.float32, 608, 2816, 768, 1), (np.float16, 2048, 1856, 2688, 0), (np.float16, 2304, 1984, 2048, 0),
                                               (np.float16, 2048, 1856, 960, 1), (np.float16, 3072, 3584, 744, 1)])
def test_matmul(dtype, R, I, O, shared):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R)
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    sparse = lambda *s: (ints(r, s, 2) * (r.random(s) < 0.25)).astype(np.float32)
    x, y, dz = sparse(R, I), sparse(I, O), sparse(R, O)
    wx, wy = dz @ y.T, x.T @ dz
    assert max(np.abs(wx).max(), np.abs(wy).max()) < 2048
    x, y, dz = (t.astype(dtype) for t in (x, y, dz))
    nb = lib.d8_matmul_scratch_bytes(dt, 3, 1, R, I, 1, I, O)
    dx, dy, dd, ws = DeviceArray.from_numpy(x), DeviceArray.from_numpy(y), DeviceArray.from_numpy(dz), DeviceArray((max(nb, 16),), np.uint8)
    gx, gy = DeviceArray.from_numpy(np.full(x.shape, np.nan, dtype)), DeviceArray.from_numpy(np.full(y.shape, np.nan, dtype))
    launches = lambda: lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches()
    before = launches()
    check(lib.d8_matmul_grad_xy(dt, dx.ptr, gx.ptr, 1, R, I, dy.ptr, gy.ptr, 1, I, O, dd.ptr, 3, ws.ptr, nb, None))
    assert launches() - before == shared
    assert np.array_equal(gx.numpy(), wx.astype(dtype)) and np.array_equal(gy.numpy(), wy.astype(dtype))


@pytest.mark.parametrize("B,size,IC,OC,F,shared", [(2, 97, 384, 192, 1, 0), (7, 35, 64, 64, 5, 1)])
def test_conv2d(oracle_port, B, size, IC, OC, F, shared):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    image, filt, geo = (B, size, size, IC), (OC, F, F), (1, 1, 1, 1, 1)
    r = rng(size)
    x, w, dz = (ints(r, s, 3).astype(np.float32) for s in (image, filt + (IC,), (B, size, size, OC)))
    nb = lib.d8_conv2d_scratch_bytes(capi.FLOAT32, 3, *image, *filt, *geo)
    dx, dw, dd, ws = DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), DeviceArray.from_numpy(dz), DeviceArray((max(nb, 16),), np.uint8)
    gx, gw = DeviceArray.from_numpy(np.full(x.shape, np.nan, np.float32)), DeviceArray.from_numpy(np.full(w.shape, np.nan, np.float32))
    before = lib.d8_conv_grad_crowded_pair_launches()
    check(lib.d8_conv2d_grad_xy(capi.FLOAT32, dx.ptr, gx.ptr, *image, dw.ptr, gw.ptr, *filt, dd.ptr, *geo, 3, ws.ptr, nb, None))
    assert lib.d8_conv_grad_crowded_pair_launches() - before == shared
    if F == 1:
        wx, ww = dz.reshape(-1, OC) @ w.reshape(OC, IC), dz.reshape(-1, OC).T @ x.reshape(-1, IC)
    else:
        wx, ww = oracle_port.conv2d_grad_x(x, w, dz, *geo), oracle_port.conv2d_grad_y(x, w, dz, *geo)
    assert np.array_equal(gx.numpy().ravel(), wx.ravel()) and np.array_equal(gw.numpy().ravel(), ww.ravel())
