"""Half products whose operands go straight into LDS: fewer K steps than stages, odd and even numbers of steps, last steps that K
cuts short, outputs of one tile and at the edges of all tiles, numbers of tiles that the XCDs share unevenly.  Integers, bit for
bit; what lies around the operands is NaN."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu

# M, N: one tile of 64 x 64, 64 x 128, 128 x 64 and 128 x 128; their edges; 15 and 273 tiles
OUTPUTS = [(64, 128), (128, 64), (264, 200), (520, 648), (136, 1048), (1672, 2632)]
STEPS = [8, 64, 72, 128, 192, 200, 256, 320, 328, 640]


@pytest.mark.parametrize("M,N", OUTPUTS)
@pytest.mark.parametrize("K", STEPS)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_products(oracle_port, M, N, K, ta, tb):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(M + 3 * N + 7 * K)
    A, B = ints(r, (K, M) if ta else (M, K), 2), ints(r, (N, K) if tb else (K, N), 2)
    want = oracle_port.gemm(ta, tb, A, B)
    assert want.max() < 2048

    def framed(a):  # 64 NaN before and after
        nan = np.full(64, np.nan, np.float16)
        d = DeviceArray.from_numpy(np.concatenate([nan, a.astype(np.float16).ravel(), nan]))
        return d, d.ptr + 128
    dA, pA = framed(A)
    dB, pB = framed(B)
    asked = lib.d8_gemm_workspace_bytes(capi.FLOAT16, ta, tb, M, N, K, 1, 0)
    for nb in {0, asked}:
        dC, ws = DeviceArray.from_numpy(np.full((M, N), np.nan, np.float16)), DeviceArray((max(nb, 16),), np.uint8)
        check(lib.d8_gemm(capi.FLOAT16, ta, tb, M, N, K, pA, A.shape[1], 0, pB, B.shape[1], 0, 0.0, dC.ptr, N, 0, 1,
                          ws.ptr if nb else None, nb, None))
        assert np.array_equal(f(dC.numpy()), want), nb
