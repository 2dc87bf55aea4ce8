"""Sums over the middle axis in chunks, whose second launch takes one, four or sixteen chunks a lane at a time and, of up to four
columns, several rows of the output in a block: on both sides of those lines.  Integers, so every order of additions gives the same; L2 norms against float64."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,C", [(1, 1), (3, 1), (5, 2), (2, 15), (3, 16), (2, 17), (17, 3), (33, 4), (9, 5), (300, 1)])
@pytest.mark.parametrize("chunks", [2, 16, 17, 64, 65, 256, 257, 321])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_chunks(K, C, chunks, dtype):
    from deep8_amd import ops
    R = 64 * chunks - 3
    if K * R * C > 8e6:
        R = 200
    r = rng(K * 100 + C + chunks)
    dz = (r.integers(-1, 2, (K, R, C), dtype=np.int8) * (r.random((K, R, C)) < 0.05)).astype(dtype)
    g = ints(r, (K, 1, C), 3).astype(dtype)
    want = dz.astype(np.float32).sum(axis=1, keepdims=True) + g.astype(np.float32)
    assert np.abs(want).max() < 2048
    assert np.array_equal(ops.add_grad(g, dz), want.astype(dtype))


@pytest.mark.parametrize("B,n", [(1, 65), (15, 1436), (24, 771), (2, 20000), (3, 64 * 257), (70000, 66)])
def test_norms(B, n):
    import ctypes
    from deep8_amd import capi
    lib = capi.init()
    x = rng(B + n).standard_normal((B, n), dtype=np.float32)
    gd, zd = (ctypes.c_int * 5)(B, 1, 1, 1, 1), (ctypes.c_int * 5)(B, 1, 1, 1, n)
    nb = lib.d8_add_grad_scratch_bytes(capi.FLOAT32, gd, zd)
    dx, dy, ws = capi.DeviceArray.from_numpy(x), capi.DeviceArray((B,)), capi.DeviceArray((max(nb, 16),), np.uint8)
    capi.check(lib.d8_l2norm(capi.FLOAT32, dx.ptr, dy.ptr, B, n, ws.ptr, nb, None))
    want = np.sqrt((x.astype(np.float64) ** 2).sum(axis=1))
    # a sum of n squares, none negative: at most n additions' roundings, in trees of at most 64 + 64 + 48 steps here
    assert np.abs(dy.numpy() - want).max() <= 180 * 2.0 ** -24 * want.max()
