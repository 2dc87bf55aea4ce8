"""d8_bias_relu_grad where only z or dz starts at an odd element: reals, so the order of the additions shows.  The sums are bit for
bit those of d8_add_grad on dpre, which is aligned and takes 16 bytes at a time."""
import ctypes

import numpy as np
import pytest

from util import nrm, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 40, 130, 256, 700])
@pytest.mark.parametrize("cols", [4, 8, 64, 128, 256, 1032])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("before", [(1, 0), (0, 1), (3, 2)])
def test_sums_are_those_of_add_grad(rows, cols, dtype, before):
    from deep8_amd import capi
    lib = capi.init()
    r = rng(rows * 3000 + cols)
    dt = capi.FLOAT32 if dtype == np.float32 else capi.FLOAT16
    z, dz = np.maximum(nrm(r, (rows, cols)), 0).astype(dtype), nrm(r, (rows, cols)).astype(dtype)
    lay = lambda v, n: capi.DeviceArray.from_numpy(np.concatenate([np.full(n, np.nan, dtype), v.ravel(), np.full(16, np.nan, dtype)]))
    dev = lay(z, before[0]), lay(dz, before[1])
    at = [d.ptr + n * z.itemsize for d, n in zip(dev, before)]
    dpre, g, h = lay(np.zeros_like(dz), 0), lay(np.zeros(cols, dtype), 0), lay(np.zeros(cols, dtype), 0)
    gd, zd = (ctypes.c_int * 5)(1, 1, 1, 1, cols), (ctypes.c_int * 5)(1, 1, 1, rows, cols)
    nb = max(lib.d8_add_grad_scratch_bytes(dt, gd, zd), 16)
    ws = capi.DeviceArray((nb,), np.uint8)
    capi.check(lib.d8_bias_relu_grad(dt, at[0], at[1], dpre.ptr, g.ptr, rows, cols, 0, ws.ptr, nb, None))
    capi.check(lib.d8_add_grad_overwrite(dt, h.ptr, gd, dpre.ptr, zd, ws.ptr, nb, None))
    assert np.array_equal(dpre.numpy()[:dz.size].reshape(dz.shape), np.where(z > 0, dz, 0).astype(dtype))
    assert np.array_equal(g.numpy()[:cols], h.numpy()[:cols])
    assert np.isnan(dpre.numpy()[dz.size:]).all() and np.isnan(g.numpy()[cols:]).all()
