"""A half MatrixMultiply whose rows start anywhere, forward, on copies of the operands with rows of whole pieces: every remainder of
a row's last piece, batches, square products, tensors that start at any element, with bias and ReLu, with room for the copies and
without.  Integers, bit for bit; what lies around the tensors is NaN; the calls that ran on copies are counted."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


def _lay(a, before):
    """the tensor `before` elements into an allocation of NaN"""
    from deep8_amd.capi import DeviceArray
    d = DeviceArray.from_numpy(np.concatenate([np.full(before, np.nan, np.float16), a.astype(np.float16).ravel(), np.full(64, np.nan, np.float16)]))
    return d, d.ptr + 2 * before


SHAPES = [(1, 300, 640, 1, 128 + n) for n in range(1, 8)] + [(1, 300, 512 + n, 1, 136) for n in (1, 3, 7)] + \
         [(1, 1000, 521, 1, 1001), (3, 150, 330, 3, 203), (2, 515, 131, 1, 645), (1, 260, 1100, 3, 257), (1, 2600, 200, 1, 2049), (1, 129, 4001, 1, 130), (1, 515, 515, 1, 515),
          (3, 203, 203, 3, 203)]


@pytest.mark.parametrize("xb,R,I,yb,O", SHAPES)
@pytest.mark.parametrize("before", [(0, 0), (1, 3)])
@pytest.mark.parametrize("copies", ["0", "1", None])
def test_forward(monkeypatch, xb, R, I, yb, O, before, copies):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    sparse = lambda s: ints(r, s, 2) * (r.random(s) < 0.5)
    x, y, bias = sparse((xb, R, I)), sparse((yb, I, O)), ints(r, (O,), 9) - 200
    z = np.matmul(x, y)
    zb = max(xb, yb)
    assert z.max() < 2040
    monkeypatch.setenv("D8_GEMM_PACK", "0")
    plain = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 0, xb, R, I, yb, I, O)
    if copies is None:
        monkeypatch.delenv("D8_GEMM_PACK")
    else:
        monkeypatch.setenv("D8_GEMM_PACK", copies)
    asked = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 0, xb, R, I, yb, I, O)
    assert asked > plain if copies == "1" else asked == plain if copies == "0" else True
    for nb in (0, plain, asked, asked + (1 << 23)):
        dx, dy = _lay(x, before[0]), _lay(y, before[1])
        db = DeviceArray.from_numpy(bias.astype(np.float16))
        ws = DeviceArray.from_numpy(np.full(max(nb, 16), 0xff, np.uint8))
        for relu in (None, 0, 1):
            dz = _lay(np.full((zb, R, O), 7), 0)
            count = lib.d8_matmul_copied_calls()
            if relu is None:
                check(lib.d8_matmul(capi.FLOAT16, dx[1], xb, R, I, dy[1], yb, I, O, dz[1], ws.ptr if nb else None, nb, None))
                want = z
            else:
                check(lib.d8_matmul_bias_relu(capi.FLOAT16, dx[1], xb, R, I, dy[1], yb, I, O, db.ptr, relu, dz[1], ws.ptr if nb else None, nb, None))
                want = z + bias
                want = np.maximum(want, 0) if relu else want
            count = lib.d8_matmul_copied_calls() - count
            if nb <= plain or copies == "0":
                assert count == 0, (nb, relu)
            elif copies == "1" and (nb > asked or not any(before)):  # (at odd addresses more may be copied than was asked for)
                assert count == 1, (nb, relu)
            got = f(dz[0].numpy())
            assert np.array_equal(got[:want.size].reshape(want.shape), want), (nb, relu)
            assert np.isnan(got[want.size:]).all(), (nb, relu)
