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


# R, I, O, forced, copied: products that do not share a launch
@pytest.mark.parametrize("R,I,O,forced,copied", [(913, 6859, 177, False, 0),    # (copies took it from 26 to 37 us)
                                                 (6539, 1674, 785, False, 1),
                                                 (5200, 1301, 1304, True, 1),   # only the second gradient has an operand to copy
                                                 (66, 3167, 528, False, 0)])    # (likewise; copies in one launch: from 13 to 16 us)
def test_products_one_after_the_other(monkeypatch, R, I, O, forced, copied):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r = rng(R + I + O)
    dx, dy, dz = (DeviceArray.from_numpy(t.astype(np.float16)) for t in (ints(r, (R, I), 2), ints(r, (I, O), 2), ints(r, (R, O), 2) * (r.random((R, O)) < 0.25)))
    left = []
    for switch in ("1" if forced else None, "0"):
        if switch is None:
            monkeypatch.delenv("D8_GEMM_PACK", raising=False)
        else:
            monkeypatch.setenv("D8_GEMM_PACK", switch)
        nb = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 3, 1, R, I, 1, I, O)
        gx, gy, ws = DeviceArray.from_numpy(np.full((R, I), np.nan, np.float16)), DeviceArray.from_numpy(np.full((I, O), np.nan, np.float16)), DeviceArray((max(nb, 16),), np.uint8)
        before = lib.d8_matmul_grad_copied_calls(), lib.d8_matmul_grad_pair_launches()
        check(lib.d8_matmul_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, 1, R, I, dy.ptr, gy.ptr, 1, I, O, dz.ptr, 3, ws.ptr if nb else None, nb, None))
        assert (lib.d8_matmul_grad_copied_calls(), lib.d8_matmul_grad_pair_launches()) == (before[0] + (copied if switch != "0" else 0), before[1])
        left.append((f(gx.numpy()), f(gy.numpy())))
    assert max(left[1][0].max(), left[1][1].max()) < 2048
    assert np.array_equal(left[0][0], left[1][0]) and np.array_equal(left[0][1], left[1][1])


def test_copies_leave_room_for_the_pieces(monkeypatch):
    """scratch for the copies alone: the products keep it for their partial sums"""
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    R, I, O = 2048, 520, 501
    q = lambda which: lib.d8_matmul_scratch_bytes(capi.FLOAT16, which, 1, R, I, 1, I, O)
    monkeypatch.setenv("D8_GEMM_PACK", "1")
    asked, largest = q(3), max(q(1), q(2))
    monkeypatch.setenv("D8_GEMM_PACK", "0")
    copies = asked - q(3)
    assert copies > 0 and largest > 0
    monkeypatch.setenv("D8_GEMM_PACK", "1")
    dx, gx, dy, gy, dz, ws = (DeviceArray((n,), np.uint8) for n in (2 * R * I, 2 * R * I, 2 * I * O, 2 * I * O, 2 * R * O, asked))
    for nb, copied in ((copies, 0), (copies + largest - 16, 0), (copies + largest, 1), (asked, 1)):
        before = lib.d8_matmul_grad_copied_calls()
        check(lib.d8_matmul_grad_xy(capi.FLOAT16, dx.ptr, gx.ptr, 1, R, I, dy.ptr, gy.ptr, 1, I, O, dz.ptr, 3, ws.ptr, nb, None))
        assert lib.d8_matmul_grad_copied_calls() - before == copied, nb
