"""Both gradients of a half MatrixMultiply whose rows start anywhere, on copies of the operands with rows of whole pieces: odd rows,
columns and inner sizes, batches (with an operand of their own and a shared one), tensors that start at any element, with room for
the copies and without, added and written.  Integers, bit for bit; what lies around the tensors is NaN; the calls that ran on copies
are counted."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu

@pytest.fixture(params=["0", "1", None])
def copies(request, monkeypatch):
    """never, always, where it is expected to pay"""
    if request.param is None:
        monkeypatch.delenv("D8_GEMM_PACK", raising=False)
    else:
        monkeypatch.setenv("D8_GEMM_PACK", request.param)
    return request.param


def _lay(a, before):
    """the tensor `before` elements into an allocation of NaN"""
    from deep8_amd.capi import DeviceArray
    d = DeviceArray.from_numpy(np.concatenate([np.full(before, np.nan, np.float16), a.astype(np.float16).ravel(), np.full(64, np.nan, np.float16)]))
    return d, d.ptr + 2 * before


SMALL = [(1, 300, 256, 1, 201), (1, 129, 200, 1, 128), (1, 201, 201, 1, 201)]  # (one of the two on the small-product kernel: no copies)
COPIED = [(1, 515, 333, 1, 77), (3, 100, 136, 3, 65), (2, 257, 131, 1, 130), (1, 2048, 520, 1, 501), (1, 130, 333, 3, 136), (1, 64, 1001, 1, 65),
          (1, 600, 520, 1, 333), (1, 261, 1030, 1, 300), (4, 300, 203, 1, 201)]


@pytest.mark.parametrize("xb,R,I,yb,O", SMALL + COPIED)
@pytest.mark.parametrize("overwrite", [0, 3])
@pytest.mark.parametrize("before", [(0, 0, 0, 0, 0), (1, 0, 0, 2, 0), (0, 3, 1, 1, 5)])
def test_gradients(oracle_port, copies, xb, R, I, yb, O, overwrite, before):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    zb = max(xb, yb)
    x, y, dz = ints(r, (xb, R, I), 2), ints(r, (yb, I, O), 2), ints(r, (zb, R, O), 2)
    gx, gy = ints(r, x.shape, 3), ints(r, y.shape, 3)
    keep = 0 if overwrite else 1
    wx = oracle_port.matmul_grad_x(x, y, dz) + keep * gx
    wy = oracle_port.matmul_grad_y(x, y, dz) + keep * gy
    assert max(wx.max(), wy.max()) < 2040
    asked = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 3, xb, R, I, yb, I, O)
    for nb in (0, asked // 2 // 16 * 16, asked, asked + (1 << 23)):
        bufs = [_lay(t, n) for t, n in zip((x, gx, y, gy, dz), before)]
        p, ws = [b[1] for b in bufs], DeviceArray((max(nb, 16),), np.uint8)
        count = lib.d8_matmul_grad_copied_calls()
        check(lib.d8_matmul_grad_xy(capi.FLOAT16, p[0], p[1], xb, R, I, p[2], p[3], yb, I, O, p[4], overwrite, ws.ptr if nb else None, nb, None))
        count = lib.d8_matmul_grad_copied_calls() - count
        if nb == 0 or copies == "0" or (xb, R, I, yb, O) in SMALL:
            assert count == 0, nb
        elif copies == "1" and (nb > asked or (nb == asked and not any(before))):  # (at odd addresses more may be copied than was asked for)
            assert count == 1, nb
        for i, want in ((1, wx), (3, wy)):
            got = f(bufs[i][0].numpy())
            assert np.array_equal(got[before[i]:before[i] + want.size].reshape(want.shape), want), (nb, i)
            assert np.isnan(got[:before[i]]).all() and np.isnan(got[before[i] + want.size:]).all()
