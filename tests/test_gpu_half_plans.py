"""Half products whose tile is chosen by the time that each takes: shapes on both sides of the choice, in whatever number of pieces
the scratch allows, with edges in every dimension.  Integers, bit for bit."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(218, 64, 1328), (1504, 3648, 128), (129, 136, 136), (513, 1032, 520), (1000, 256, 1000), (2040, 72, 968), (96, 4096, 200),
                                   (3000, 192, 72), (640, 1152, 640)])
@pytest.mark.parametrize("trans", [(0, 0), (0, 1), (1, 0)])
def test_pieces_that_fit(M, K, N, trans):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(M + K + N)
    A = ints(r, (M, K), 2) * (r.random((M, K)) < 0.25)
    B = ints(r, (K, N), 2) * (r.random((K, N)) < 0.25)
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.abs(want).max() < 2048
    tA, tB = trans
    dA = DeviceArray.from_numpy(np.ascontiguousarray((A.T if tA else A).astype(np.float16)))
    dB = DeviceArray.from_numpy(np.ascontiguousarray((B.T if tB else B).astype(np.float16)))
    for pieces in (0, 1, 2, 3, 5, 8, 40):
        nb = pieces * M * N * 4
        ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
        dC = DeviceArray.from_numpy(np.full((M, N), np.nan, np.float16))
        check(lib.d8_gemm(capi.FLOAT16, tA, tB, M, N, K, dA.ptr, M if tA else K, 0, dB.ptr, K if tB else N, 0, 0.0, dC.ptr, N, 0, 1, ws.ptr if nb else None, nb, None))
        assert np.array_equal(dC.numpy().astype(np.float64), want), pieces


@pytest.mark.parametrize("R,I,O", [(128, 1664, 2752), (3968, 1712, 96)])
def test_forward_products_that_run_whole(R, I, O):
    """more than 4 MB of operands: by 64 x 64 tiles in one pass, so nothing is written to the scratch"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    x, y = (ints(r, s, 2) * (r.random(s) < 0.25) for s in ((R, I), (I, O)))
    z = x.astype(np.float32) @ y.astype(np.float32)
    assert np.abs(z).max() < 2048
    nb = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 0, 1, R, I, 1, I, O)
    dx, dy, ws = DeviceArray.from_numpy(x.astype(np.float16)), DeviceArray.from_numpy(y.astype(np.float16)), DeviceArray.from_numpy(np.full(nb // 4, np.nan, np.float32))
    dz = DeviceArray.from_numpy(np.full(z.shape, np.nan, np.float16))
    check(lib.d8_matmul(capi.FLOAT16, dx.ptr, 1, R, I, dy.ptr, 1, I, O, dz.ptr, ws.ptr, nb, None))
    assert nb > 0 and np.isnan(ws.numpy()).all()
    assert np.array_equal(dz.numpy(), z.astype(np.float16))
