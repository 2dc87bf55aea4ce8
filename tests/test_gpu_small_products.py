"""Products small enough for one load latency: reductions at the ends of a chunk and of what the waves share, sums of many
short products (their chunks count one by one), bias and ReLu in the store."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


# a sum of `red` products of K columns each; the last ones have 64 chunks in all
@pytest.mark.parametrize("M,N,K,red", [(33, 65, 1, 1), (64, 256, 128, 1), (31, 32, 63, 1), (50, 40, 512, 1), (20, 70, 16, 5), (32, 32, 8, 64), (40, 33, 5, 37)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_small_products(oracle_port, M, N, K, red, ta, tb, dtype):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt, es = capi.dtype_id(np.dtype(dtype)), np.dtype(dtype).itemsize
    r = rng(M + N + K + red)
    A, B = ints(r, (red,) + ((K, M) if ta else (M, K)), 3), ints(r, (red,) + ((N, K) if tb else (K, N)), 3)
    want = sum(oracle_port.gemm(ta, tb, A[i], B[i]) for i in range(red))
    assert want.max() < 2048
    for start in (0, 1):  # an element into the allocation, NaN on either side
        pad = lambda a: np.concatenate([np.full(start, np.nan), a.ravel(), np.full(8, np.nan)]).astype(dtype)
        dA, dB, dC = DeviceArray.from_numpy(pad(A)), DeviceArray.from_numpy(pad(B)), DeviceArray.from_numpy(np.full((M, N), np.nan, dtype))
        check(lib.d8_gemm(dt, ta, tb, M, N, K, dA.ptr + start * es, A.shape[2], A[0].size, dB.ptr + start * es, B.shape[2], B[0].size, 0.0, dC.ptr, N,
                          0 if red > 1 else M * N, red, None, 0, None))
        assert np.array_equal(f(dC.numpy()), want), start


@pytest.mark.parametrize("rows,inner,cols", [(64, 256, 10), (37, 100, 33), (128, 512, 128)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_bias_and_relu_round_as_passes_of_their_own(rows, inner, cols, dtype):
    from deep8_amd import ops
    r = rng(rows + cols)
    x, y, b = (a.astype(dtype) for a in (r.standard_normal((1, rows, inner)), r.standard_normal((1, inner, cols)) / 8, r.standard_normal(cols)))
    want = ops.relu(ops.add(ops.matmul(x, y), b.reshape(1, cols)))
    got = ops.matmul_bias_relu(x, y, b)
    assert np.array_equal(got, want.reshape(got.shape))


@pytest.mark.parametrize("M,N", [(1, 1), (2, 1), (1, 3), (2, 2), (5, 1), (34, 103), (19, 111), (37, 175)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_long_reductions_of_few_outputs(oracle_port, M, N, dtype):
    """cut into many pieces: groups of four outputs with one, two and three left over, and fewer than four outputs in all;
    summed products that lie an odd number of elements apart (the any-shape kernel) and a single one"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt, r = capi.dtype_id(np.dtype(dtype)), rng(M + N)
    for batch, K in ((1, 9000), (51, 339)):
        A, B = ints(r, (batch, M, K), 3), ints(r, (batch, K, N), 3)
        A *= r.random(A.shape) < 0.05  # (thinned: half holds the sums)
        want = sum(oracle_port.gemm(0, 0, A[i], B[i]) for i in range(batch))
        assert 0 < want.max() < 2048
        dA, dB = DeviceArray.from_numpy(A.astype(dtype)), DeviceArray.from_numpy(B.astype(dtype))
        sC = 0 if batch > 1 else M * N
        nb = lib.d8_gemm_workspace_bytes(dt, 0, 0, M, N, K, batch, sC)
        dC, ws = DeviceArray.from_numpy(np.full((M, N), np.nan, dtype)), DeviceArray.from_numpy(np.full(nb + 64, 255, np.uint8))
        check(lib.d8_gemm(dt, 0, 0, M, N, K, dA.ptr, K, M * K, dB.ptr, N, K * N, 0.0, dC.ptr, N, sC, batch, ws.ptr, nb, None))
        assert np.array_equal(dC.numpy().astype(np.float32), want), batch
