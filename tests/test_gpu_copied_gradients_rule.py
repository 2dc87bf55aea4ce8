"""Both gradients of half products with odd sizes for which copies pay although each product has only a few K steps a compute unit:
they run on copies, and leave what they leave without.  Narrow ones, for which copies do not pay, run without.  Integers, bit for bit."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xb,R,I,O,copied", [(1, 3039, 376, 2289, 1), (6, 1005, 368, 1211, 1), (4, 174, 1524, 872, 1), (1, 2375, 369, 1146, 1),
                                             (1, 4288, 878, 64, 0), (58, 1888, 46, 64, 0), (1, 64, 3712, 15, 1)])
def test_calls_that_run_on_copies(monkeypatch, xb, R, I, O, copied):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    sparse = lambda s: ints(r, s, 2) * (r.random(s) < 0.25)
    dx, dy, dz = (DeviceArray.from_numpy(sparse(s).astype(np.float16)) for s in ((xb, R, I), (xb, I, O), (xb, R, O)))
    left = []
    for switch in (None, "0"):
        if switch is None:
            monkeypatch.delenv("D8_GEMM_PACK", raising=False)
        else:
            monkeypatch.setenv("D8_GEMM_PACK", switch)
        nb = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 3, xb, R, I, xb, I, O)
        gx, gy, ws = (DeviceArray.from_numpy(np.full(s, np.nan, np.float16)) for s in ((xb, R, I), (xb, I, O), (max(nb, 16) // 2,)))
        before = lib.d8_matmul_grad_copied_calls()
        check(lib.d8_matmul_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, xb, R, I, dy.ptr, gy.ptr, xb, I, O, dz.ptr, 3, ws.ptr if nb else None, nb, None))
        assert lib.d8_matmul_grad_copied_calls() - before == (copied if switch is None else 0)
        left.append((f(gx.numpy()), f(gy.numpy())))
    assert max(left[1][0].max(), left[1][1].max()) < 2048
    assert np.array_equal(left[0][0], left[1][0]) and np.array_equal(left[0][1], left[1][1])
