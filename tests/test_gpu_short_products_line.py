"""Forward products on both sides of the line that workgroups times the reduction draw for the kernel for small products (400 elements a
compute unit: 256 and 384 workgroups of 32 x 32 outputs; 240 for up to 128 rows in half, none for rows that start anywhere).  Integers
against numpy, bit for bit."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,xb,R,K,O", [(np.float16, 1, 512, K, 512) for K in (399, 400, 401, 408)] + [(np.float16, 10, 104, 736, 176), (np.float16, 1, 250, 1000, 344)] +
                         [(np.float16, 1, 128, K, 2048) for K in (232, 240, 248)] + [(np.float16, 1, 129, 248, 1632), (np.float16, 1, 64, 832, 1920), (np.float16, 2, 64, 1000, 64)] +
                         [(np.float16, 1, 512, K, 511) for K in (399, 400, 405)] + [(np.float16, 43, 64, 704, 34), (np.float16, 1, 77, 1021, 2047)] +
                         [(np.float32, 1, 512, K, 760) for K in (265, 266, 267, 268)] + [(np.float32, 1, 512, 512, 512), (np.float32, 13, 112, 496, 152)])
def test_forward(dtype, xb, R, K, O):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + K + O)
    x, y = (ints(r, s, 2) * (r.random(s) < 0.7) for s in ((xb, R, K), (xb, K, O)))
    z = np.matmul(x.astype(np.float32), y.astype(np.float32))
    assert z.max() < 2048
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    dx, dy = DeviceArray.from_numpy(x.astype(dtype)), DeviceArray.from_numpy(y.astype(dtype))
    nb = lib.d8_matmul_scratch_bytes(dt, 0, xb, R, K, xb, K, O)
    ws, dz = DeviceArray((max(nb, 16),), np.uint8), DeviceArray.from_numpy(np.full(z.size + 64, np.nan, dtype))
    check(lib.d8_matmul(dt, dx.ptr, xb, R, K, dy.ptr, xb, K, O, dz.ptr, ws.ptr if nb else None, nb, None))
    got = f(dz.numpy())
    assert np.array_equal(got[:z.size].reshape(z.shape), z) and np.isnan(got[z.size:]).all()
