"""Products whose rows start anywhere: odd leading dimensions, odd reductions, pointers that are only aligned to an element,
batches with odd strides.  The operands lie inside buffers full of NaN (what a piece brings in from past a row's end must
never reach a result), C inside a buffer whose other elements must survive.  Integers, bit for bit."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


def _embed(a, ld, first, total_rows_gap, dtype):
    """a [batch][rows][cols] as rows of leading dimension ld, `first` elements into a buffer of NaN, `gap` elements between
    the batch's matrices; returns buffer, stride of the batch"""
    b, rows, cols = a.shape
    stride = rows * ld + total_rows_gap
    buf = np.full(first + b * stride + 9, np.nan, dtype)
    for i in range(b):
        for r in range(rows):
            at = first + i * stride + r * ld
            buf[at:at + cols] = a[i, r]
    return buf, stride


# M, N, K: tile edges (64, 128), remainders of a 16-byte piece, of a dword and of a K step, fewer rows than any tile
SHAPES = [(130, 127, 65), (64, 129, 333), (200, 33, 515), (37, 41, 1031), (128, 128, 129), (1, 300, 700), (257, 1, 640), (129, 255, 7)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_rows_that_start_anywhere(oracle_port, M, N, K, ta, tb, dtype):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt, es = capi.dtype_id(np.dtype(dtype)), np.dtype(dtype).itemsize
    r = rng(M + 3 * N + 7 * K + ta + 2 * tb)
    hi = 2 if dtype == np.float16 else 9
    for batch, pad, first, gap, workspace in ((1, 0, 0, 0, True), (1, 3, 1, 0, False), (3, 0, 1, 1, True), (2, 1, 2, 0, True)):
        A = ints(r, (batch,) + ((K, M) if ta else (M, K)), hi)
        B = ints(r, (batch,) + ((N, K) if tb else (K, N)), hi)
        C = ints(r, (batch, M, N), 5)
        lda, ldb, ldc = A.shape[2] + pad, B.shape[2] + 2 * pad, N + pad
        bufA, sA = _embed(A, lda, first, gap, dtype)
        bufB, sB = _embed(B, ldb, first, gap, dtype)
        bufC, sC = _embed(C, ldc, first, gap, dtype)
        dA, dB, dC = (DeviceArray.from_numpy(v) for v in (bufA, bufB, bufC))
        nb = lib.d8_gemm_workspace_bytes(dt, ta, tb, M, N, K, batch, sC) if workspace else 0
        ws = DeviceArray((max(nb, 16),), np.uint8)
        check(lib.d8_gemm(dt, ta, tb, M, N, K, dA.ptr + first * es, lda, sA, dB.ptr + first * es, ldb, sB, 1.0, dC.ptr + first * es, ldc, sC,
                          batch, ws.ptr if nb else None, nb, None))
        want = np.stack([oracle_port.gemm(ta, tb, A[i], B[i]) for i in range(batch)]) + C
        assert dtype == np.float32 or want.max() < 2048
        wantbuf, _ = _embed(want, ldc, first, gap, dtype)
        assert np.array_equal(f(dC.numpy()), f(wantbuf), equal_nan=True), (batch, pad, first, gap)


@pytest.mark.parametrize("M,N,K", [(2310, 1930, 7), (2310, 1930, 16), (2310, 1930, 17), (2310, 1930, 33), (2310, 1930, 65), (2310, 1930, 81), (4230, 65, 3)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_short_products_over_many_tiles(oracle_port, M, N, K, ta, tb, dtype):
    """either side of the reductions and outputs that are left to the any-shape kernel; a sum of products too"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt = capi.dtype_id(np.dtype(dtype))
    r = rng(M + N + K)
    batch = 8 if N == 65 else 2 if K > 17 else 4 if (ta, dtype) == (1, np.float16) else 1
    hi = 5 if K > 17 else 9
    A, B = ints(r, (batch,) + ((K, M) if ta else (M, K)), hi), ints(r, (batch,) + ((N, K) if tb else (K, N)), hi)
    (bufA, sA), (bufB, sB) = _embed(A, A.shape[2], 0, 0, dtype), _embed(B, B.shape[2], 0, 0, dtype)
    dA, dB = DeviceArray.from_numpy(bufA), DeviceArray.from_numpy(bufB)
    each = [oracle_port.gemm(ta, tb, A[i], B[i]) for i in range(batch)]
    for summed in (False, True) if N == 65 and K % 2 else (False,):
        want = sum(each) if summed else np.stack(each)
        assert want.max() < 2048
        dC = DeviceArray.from_numpy(np.full(want.shape, np.nan, dtype))
        sC = 0 if summed else M * N
        nb = lib.d8_gemm_workspace_bytes(dt, ta, tb, M, N, K, batch, sC)
        ws = DeviceArray((max(nb, 16),), np.uint8)
        check(lib.d8_gemm(dt, ta, tb, M, N, K, dA.ptr, A.shape[2], sA, dB.ptr, B.shape[2], sB, 0.0, dC.ptr, N, sC, batch, ws.ptr if nb else None,
                          nb, None))
        assert np.array_equal(f(dC.numpy()), want)


@pytest.mark.parametrize("batch,stride_odd", [(5, False), (4, True)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_summed_batch_of_odd_matrices(oracle_port, batch, stride_odd, dtype):
    """strideC = 0: all products of the batch in one sum; half matrices an odd number of elements apart change a row's
    parity from product to product"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    dt = capi.dtype_id(np.dtype(dtype))
    M, N, K = 131, 77, 67
    r = rng(batch)
    A, B = ints(r, (batch, K, M), 2), ints(r, (batch, K, N), 2)
    gap = 1 if stride_odd == (K * M % 2 == 0) else 0
    gapB = 1 if stride_odd == (K * N % 2 == 0) else 0
    (bufA, sA), (bufB, sB) = _embed(A, M, 0, gap, dtype), _embed(B, N, 0, gapB, dtype)
    assert sA % 2 == sB % 2 == int(stride_odd)
    dA, dB, dC = DeviceArray.from_numpy(bufA), DeviceArray.from_numpy(bufB), DeviceArray((M, N), dtype, zero=True)
    nb = lib.d8_gemm_workspace_bytes(dt, 1, 0, M, N, K, batch, 0)
    ws = DeviceArray((max(nb, 16),), np.uint8)
    check(lib.d8_gemm(dt, 1, 0, M, N, K, dA.ptr, M, sA, dB.ptr, N, sB, 0.0, dC.ptr, N, 0, batch, ws.ptr, nb, None))
    want = sum(oracle_port.gemm(1, 0, A[i], B[i]) for i in range(batch))
    assert want.max() < 2048 and np.array_equal(f(dC.numpy()), want)


@pytest.mark.parametrize("rows,inner,cols", [(200, 72, 77), (1030, 64, 130), (96, 1000, 333), (2310, 13, 1931)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_bias_and_relu_of_odd_columns_round_as_passes_of_their_own(rows, inner, cols, dtype):
    """matmul_bias_relu on rows that start anywhere: bit for bit matmul, add, relu -- in half too, where the product is
    rounded before the bias is added"""
    from deep8_amd import ops
    r = rng(rows + cols)
    c = lambda a: a.astype(dtype)
    x, y, b = c(r.standard_normal((1, rows, inner))), c(r.standard_normal((1, inner, cols)) / 8), c(r.standard_normal(cols))
    want = ops.relu(ops.add(ops.matmul(x, y), b.reshape(1, cols)))
    got = ops.matmul_bias_relu(x, y, b)
    assert np.array_equal(got, want.reshape(got.shape))
