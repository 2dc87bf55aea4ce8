"""Passes over partial sums: any number of pieces (the loads in flight at once are two, four or eight a thread, those past the
last piece zeros), outputs whose last group of four is short, and column sums around the chunks' and the lanes' sizes.  Integers,
so every order of additions gives the same.  A limit on the scratch is not the number of pieces: where that matters, the pieces that
were written are counted."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


# M x N outputs in a thread row per piece (few outputs) and a thread per group (more than 196608 outputs, at most 8 pieces)
@pytest.mark.parametrize("M,N,K,pieces", [(64, 128, 4096, n) for n in (2, 7, 8, 9, 16, 17, 31, 32, 33, 47)] +
                         [(1, 1, 4096, 5), (1, 3, 4096, 9), (3, 67, 4096, 17), (65, 101, 4096, 33)] +
                         [(512, 512, 2048, n) for n in (2, 3, 4, 5, 8)] + [(511, 513, 2048, 5)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_pieces_of_a_product(M, N, K, pieces, dtype):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(M + N + pieces)
    A = (ints(r, (K, M), 2) * (r.random((K, M)) < 0.25)).astype(dtype)
    B = (ints(r, (K, N), 2) * (r.random((K, N)) < 0.25)).astype(dtype)
    C0 = ints(r, (M, N), 3).astype(dtype)
    want = A.astype(np.float64).T @ B.astype(np.float64)
    assert np.abs(want).max() + 3 < 2048
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    dA, dB = DeviceArray.from_numpy(A), DeviceArray.from_numpy(B)
    ws = DeviceArray.from_numpy(np.full(pieces * M * N + 8, np.nan, np.float32))
    for beta, expected in ((0.0, want), (1.0, want + C0)):
        dC = DeviceArray.from_numpy(C0)
        check(lib.d8_gemm(dt, 1, 0, M, N, K, dA.ptr, M, 0, dB.ptr, N, 0, beta, dC.ptr, N, 0, 1, ws.ptr, pieces * M * N * 4, None))
        assert np.array_equal(dC.numpy(), expected.astype(dtype)), beta


# pieces taken: a thread row per piece with two, four and eight loads in flight, one round and two of eight; a thread per group with
# four and eight, whole groups of four outputs in a row and not
@pytest.mark.parametrize("dtype,M,N,K,pieces", [(np.float32, 64, 128, 16384, n) for n in (2, 17, 31, 32, 47, 64, 128)] +
                         [(np.float16, 64, 128, 32768, n) for n in (9, 17, 31, 47, 64, 86)] +
                         [(np.float32, 3, 67, 16384, 47), (np.float16, 65, 101, 32768, 64)] +
                         [(np.float32, 512, 768, 4096, n) for n in (2, 5, 8)] + [(np.float16, 512, 768, 4096, n) for n in (2, 4, 5, 6, 7, 8)] +
                         [(np.float32, 511, 513, 4096, n) for n in (3, 7)] + [(np.float16, 511, 513, 4096, n) for n in (3, 4, 5, 8)])
def test_pieces_taken(dtype, M, N, K, pieces):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(M + N + pieces)
    A = (ints(r, (K, M), 2) * (r.random((K, M)) < 0.1)).astype(np.float32)
    B = (ints(r, (K, N), 2) * (r.random((K, N)) < 0.1)).astype(np.float32)
    want = A.T @ B
    assert np.abs(want).max() < 2048
    dt = capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32
    dA, dB = DeviceArray.from_numpy(A.astype(dtype)), DeviceArray.from_numpy(B.astype(dtype))
    ws = DeviceArray.from_numpy(np.full((pieces + 1) * M * N, np.nan, np.float32))
    dC = DeviceArray.from_numpy(np.full((M, N), np.nan, dtype))
    check(lib.d8_gemm(dt, 1, 0, M, N, K, dA.ptr, M, 0, dB.ptr, N, 0, 0.0, dC.ptr, N, 0, 1, ws.ptr, pieces * M * N * 4, None))
    assert np.array_equal(dC.numpy(), want.astype(dtype))
    written = ~np.isnan(ws.numpy()).reshape(pieces + 1, M * N)
    assert written[:pieces].all() and not written[pieces].any()


@pytest.mark.parametrize("rows", [2, 31, 33, 64, 65, 96, 97, 129, 1000, 8193])
@pytest.mark.parametrize("cols", [1, 3, 8, 64, 255, 256, 260, 1024])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_column_sums(rows, cols, dtype):
    from deep8_amd import ops
    r = rng(rows + cols)
    dz = ((ints(r, (rows, cols), 2) - 1) * (r.random((rows, cols)) < min(1.0, 600.0 / rows))).astype(dtype)
    sums = dz.astype(np.float64).sum(axis=0)
    assert np.abs(sums).max() < 2040
    got = ops.add_grad(np.ones((1, 1, cols), dtype), dz.reshape(1, rows, cols))
    assert np.array_equal(got.reshape(cols), (sums + 1).astype(dtype))
    z = ints(r, (rows, cols), 2).astype(dtype)
    gated = np.where(z > 0, dz, 0).astype(dtype)
    dpre, db = ops.bias_relu_grad(z, dz, None, True, False)
    assert np.array_equal(dpre, gated) and np.array_equal(db, gated.astype(np.float64).sum(axis=0).astype(dtype))
