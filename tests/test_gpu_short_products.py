"""Products of short reductions on the kernel for small products: on both sides of the lines where it takes them (the reduction, the
number of 32 x 32 tiles), sizes that no tile divides, odd rows, batches, bias and ReLu.  Integers against numpy, bit for bit; what lies
behind an output is NaN."""
import numpy as np
import pytest

from util import f, ints, nrm, rng

pytestmark = pytest.mark.gpu


def _sparse(r, shape, K):
    return ints(r, shape, 2) * (r.random(shape) < min(1.0, (1000.0 / K) ** 0.5))


# K on both sides of 512 (fp32) and 1024 (half); 256 | 257 tiles (half) and 384 | 385 (fp32) of 32 x 32
FORWARD = [(1, 160, K, 1, 200) for K in (1, 7, 64, 511, 512, 513, 1016, 1023, 1024, 1025)] + \
          [(1, 512, 136, 1, 512), (1, 32 * 257, 72, 1, 32), (1, 32 * 384, 72, 1, 25), (1, 32 * 385 - 5, 40, 1, 32), (9, 131, 96, 9, 33), (9, 131, 97, 1, 35),
           (1, 96, 264, 5, 160), (5, 130, 200, 1, 161)]


@pytest.mark.parametrize("xb,R,K,yb,O", FORWARD)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_forward(xb, R, K, yb, O, dtype):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + K + O)
    x, y, bias = _sparse(r, (xb, R, K), K), _sparse(r, (yb, K, O), K), ints(r, (O,), 9) - 200
    z = np.matmul(x, y)
    assert z.max() < 2040
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    dx, dy, db = (DeviceArray.from_numpy(a.astype(dtype)) for a in (x, y, bias))
    nb = lib.d8_matmul_scratch_bytes(dt, 0, xb, R, K, yb, K, O)
    ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
    for relu in (None, 0, 1):
        dz = DeviceArray.from_numpy(np.full(z.size + 64, np.nan, dtype))
        if relu is None:
            check(lib.d8_matmul(dt, dx.ptr, xb, R, K, dy.ptr, yb, K, O, dz.ptr, ws.ptr if nb else None, nb, None))
        else:
            check(lib.d8_matmul_bias_relu(dt, dx.ptr, xb, R, K, dy.ptr, yb, K, O, db.ptr, relu, dz.ptr, ws.ptr if nb else None, nb, None))
        want = z if relu is None else np.maximum(z + bias, 0) if relu else z + bias
        got = f(dz.numpy())
        assert np.array_equal(got[:z.size].reshape(z.shape), want), relu
        assert np.isnan(got[z.size:]).all(), relu


def test_gradients_share_a_launch():
    """and a call for one of them leaves the bits of the call for both"""
    from deep8_amd import capi, ops
    lib = capi.init()
    r = rng(3)
    for dtype in (np.float32, np.float16):
        for R, I, O in ((280, 192, 64), (64, 704, 336) if dtype == np.float32 else (640, 320, 128), (336, 320, 14), (64, 511, 61)):
            x, y, dz = (nrm(r, s).astype(dtype) for s in ((1, R, I), (1, I, O), (1, R, O)))
            before = lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches()
            gx, gy = ops.matmul_grad_xy(x, y, dz, overwrite_x=True, overwrite_y=True)
            assert lib.d8_matmul_grad_pair_launches() + lib.d8_matmul_grad_kept_pair_launches() == before + 1, (R, I, O)
            assert np.array_equal(gx, ops.matmul_grad_x(x, y, dz, overwrite=True)) and np.array_equal(gy, ops.matmul_grad_y(x, y, dz, overwrite=True))
