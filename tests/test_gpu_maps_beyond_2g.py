"""im2col and col2im of 2^31 elements and more, whose indices do not fit 32 bits, also within one patch row: a filter of one row and
three columns over a wide image, so that what every element has to be follows from its neighbours.  Bit for bit (small integers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(B, H, W):
    """small integers whose pattern is no divisor of a row's length"""
    n = 1000003
    few = ((np.arange(n, dtype=np.int64) * 2654435761 >> 7) % 7 - 3).astype(np.float16)
    return np.resize(few, (B, H, W))


def test_rows_of_odd_length_gathered_side_by_side():
    from deep8_amd import capi
    lib = capi.init()
    B, H, W = 3, 1021, 233747
    x = _image(B, H, W)
    assert 3 * x.size >= 1 << 31
    dx, dcol = capi.DeviceArray.from_numpy(x), capi.DeviceArray((B, H, W, 3), np.float16)
    capi.check(lib.d8_im2col(capi.FLOAT16, dx.ptr, dcol.ptr, B, H, W, 1, H, W, 1, 3, 1, 1, 1, 1, 0, 1, None))
    col = dcol.numpy()
    for b in range(B):
        assert np.array_equal(col[b, :, :, 1], x[b])
        assert np.array_equal(col[b, :, 1:, 0], x[b, :, :-1]) and not col[b, :, 0, 0].any()
        assert np.array_equal(col[b, :, :-1, 2], x[b, :, 1:]) and not col[b, :, -1, 2].any()


def test_taps_added_into_the_image():
    from deep8_amd import capi
    lib = capi.init()
    B, H, W = 3, 1021, 701209
    im = _image(B, H, W)
    assert im.size >= 1 << 31
    col = _image(B, H, 3 * W).reshape(B, H, W, 3)
    dim, dcol = capi.DeviceArray.from_numpy(im), capi.DeviceArray.from_numpy(col)
    capi.check(lib.d8_col2im(capi.FLOAT16, dcol.ptr, dim.ptr, B, H, W, 1, H, W, 1, 3, 1, 1, 1, 1, 0, 1, None))
    got = dim.numpy()
    for b in range(B):
        im[b] += col[b, :, :, 1]
        im[b, :, :-1] += col[b, :, 1:, 0]
        im[b, :, 1:] += col[b, :, :-1, 2]
        assert np.array_equal(got[b], im[b])


@pytest.mark.parametrize("C", [(1 << 30) + 1, 1 << 30])
def test_patch_rows_beyond_31_bits(C):
    from deep8_amd import capi
    lib = capi.init()
    assert 3 * C >= 1 << 31
    x, before = _image(1, 1, C), _image(1, 1, C)[..., ::-1]
    dx, dcol, dim = capi.DeviceArray.from_numpy(x), capi.DeviceArray((3, C), np.float16), capi.DeviceArray.from_numpy(np.ascontiguousarray(before))
    geo = (1, 1, 1, C, 1, 1, 1, 3, 1, 1, 1, 1, 0, 2)  # one pixel, which only the last tap of a row of three reaches
    capi.check(lib.d8_im2col(capi.FLOAT16, dx.ptr, dcol.ptr, *geo, None))
    col = dcol.numpy()
    assert not col[:2].any() and np.array_equal(col[2], x[0, 0])
    del col
    capi.check(lib.d8_col2im(capi.FLOAT16, dcol.ptr, dim.ptr, *geo, None))
    assert np.array_equal(dim.numpy(), x + before)
