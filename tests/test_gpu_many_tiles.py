"""Half products of few K steps over more than two tiles a compute unit: the variant of two stages, of which three workgroups fit.
Whole numbers, bit for bit."""
import numpy as np
import pytest

from util import f, h, ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(128 * 513, 64), (128 * 520 + 72, 104), (64, 128 * 513), (72, 128 * 300 + 8)])
@pytest.mark.parametrize("K", [8, 64, 72, 136, 192, 264])
@pytest.mark.parametrize("tb", [0, 1])
def test_products(M, N, K, tb):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(M + 3 * N + 7 * K + tb)
    A, B = ints(r, (M, K), 2), ints(r, (N, K) if tb else (K, N), 2)
    want = A @ (B.T if tb else B)  # (fp32 holds these sums)
    assert want.max() < 2048
    dA, dB = DeviceArray.from_numpy(h(A)), DeviceArray.from_numpy(h(B))
    dC = DeviceArray.from_numpy(np.full((M, N), np.nan, np.float16))
    check(lib.d8_gemm(capi.FLOAT16, 0, tb, M, N, K, dA.ptr, K, 0, dB.ptr, B.shape[1], 0, 0.0, dC.ptr, N, 0, 1, None, 0, None))
    assert np.array_equal(f(dC.numpy()), want)


@pytest.mark.parametrize("C,OC,F", [(8, 16, 1), (8, 24, 3), (72, 40, 2), (64, 64, 2), (16, 104, 1)])
def test_conv2d(oracle_port, C, OC, F):
    from deep8_amd import ops
    r = rng(C + OC)
    x, w = ints(r, (8, 97, 95, C), 2), ints(r, (OC, F, F, C), 2)
    got = f(ops.conv2d(h(x), h(w), True))
    assert np.array_equal(got, oracle_port.conv2d(x, w, True, 1, 1, 1, 1))


@pytest.mark.parametrize("C,OC,F,s", [(8, 11, 4, 2), (8, 64, 2, 2), (72, 24, 3, 2), (64, 40, 3, 3)])
def test_deconv2d(oracle_port, C, OC, F, s):
    from deep8_amd import ops
    r = rng(C + OC)
    x, w = ints(r, (16, 37, 40, C), 2), ints(r, (OC, F, F, C), 2)
    assert np.array_equal(f(ops.deconv2d(h(x), h(w), False, s, s)), oracle_port.deconv2d(x, w, False, s, s))
