"""Gradients of a MatrixMultiply that share a launch: K steps cut short, more workgroups than the chip holds, batches.  One call for both
leaves the bits of two calls.  Integers against numpy, bit for bit."""
import numpy as np
import pytest

from util import ints, nrm, rng

pytestmark = pytest.mark.gpu


def _sparse(r, shape, K):
    return ints(r, shape, 2) * (r.random(shape) < min(1.0, (1000.0 / K) ** 0.5))


GRADIENTS = [(1, 280, 192, 1, 64), (1, 64, 704, 1, 336), (1, 512, 500, 1, 512), (1, 1024, 32, 1, 1024), (1, 1023, 33, 1, 47), (1, 1025, 33, 1, 47), (1, 64, 2525, 1, 120),
             (1, 128, 3200, 1, 64), (1, 336, 320, 1, 14), (2, 512, 224, 2, 64), (3, 150, 131, 3, 67), (5, 100, 72, 1, 200), (1, 100, 72, 5, 200),
             # tiles: K steps cut short in one or both, and more workgroups than the chip holds
             (1, 448, 1304, 1, 152), (1, 1192, 1024, 1, 72), (1, 1190, 1024, 1, 640), (4, 72, 2496, 4, 128), (1, 4104, 1536, 1, 200), (4, 1024, 512, 1, 480), (6, 520, 712, 6, 968)]


@pytest.mark.parametrize("xb,R,I,yb,O", GRADIENTS)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_gradients(xb, R, I, yb, O, dtype):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O + 1)
    zb = max(xb, yb)
    x, y, dz = _sparse(r, (xb, R, I), R * zb), _sparse(r, (yb, I, O), O * zb), _sparse(r, (zb, R, O), max(R, O) * zb)
    gx, gy = ints(r, x.shape, 3), ints(r, y.shape, 3)
    f64 = [a.astype(np.float64) for a in (x, y, dz)]
    wx, wy = np.matmul(f64[2], f64[1].transpose(0, 2, 1)), np.matmul(f64[0].transpose(0, 2, 1), f64[2])
    wx, wy = (w.sum(axis=0, keepdims=True) if a.shape[0] < zb else w for w, a in ((wx, x), (wy, y)))
    assert max(wx.max(), wy.max()) < 2040
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    asked = lib.d8_matmul_scratch_bytes(dt, 3, xb, R, I, yb, I, O)
    for nb in (0, asked // 2 // 16 * 16, asked):
        ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
        p = [DeviceArray.from_numpy(a.astype(dtype)) for a in (x, gx, y, gy, dz)]
        check(lib.d8_matmul_grad_xy(dt, p[0].ptr, p[1].ptr, xb, R, I, p[2].ptr, p[3].ptr, yb, I, O, p[4].ptr, 1, ws.ptr if nb else None, nb, None))
        assert np.array_equal(p[1].numpy(), wx.astype(dtype)) and np.array_equal(p[3].numpy(), (wy + gy).astype(dtype)), nb
    x, y, dz = (nrm(r, a.shape).astype(dtype) for a in (x, y, dz))
    before = lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches()
    gx, gy = ops.matmul_grad_xy(x, y, dz, overwrite_x=True, overwrite_y=True)
    assert lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches() - before <= 1
    assert np.array_equal(gx, ops.matmul_grad_x(x, y, dz, overwrite=True))
    assert np.array_equal(gy, ops.matmul_grad_y(x, y, dz, overwrite=True))


def test_which_gradients_share_a_launch():
    from deep8_amd import capi, ops
    lib = capi.init()
    r = rng(3)
    for dtype in (np.float32, np.float16):
        for R, I, O in ((448, 1304, 152), (1190, 1024, 640), (4104, 1536, 200)):
            x, y, dz = (nrm(r, s).astype(dtype) for s in ((1, R, I), (1, I, O), (1, R, O)))
            before = lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches()
            ops.matmul_grad_xy(x, y, dz, overwrite_x=True, overwrite_y=True)
            assert lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches() == before + 1, (R, I, O)
