"""im2col of rows whose length no 16-byte piece divides, side by side: pieces that cross taps, rows, lines of outputs and images, a last piece
that is short, and a matrix that starts anywhere.  Bit for bit against the oracle; what lies behind the matrix stays."""
import numpy as np
import pytest

from util import f, nrm, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("FH,FW,sy,sx,dy,dx", [(1, 1, 1, 1, 1, 1), (1, 3, 1, 1, 1, 1), (3, 1, 2, 1, 1, 1), (3, 3, 1, 1, 1, 1), (2, 3, 2, 3, 2, 1), (5, 5, 1, 2, 1, 1)])
@pytest.mark.parametrize("C", [1, 2, 3, 5, 7, 9, 13, 35])
@pytest.mark.parametrize("covered", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("before,many", [(0, 0), (0, 1), (1, 1)])
def test_pieces(oracle_port, FH, FW, sy, sx, dy, dx, C, covered, dtype, before, many):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    # (enough pieces for the kernel that gathers whole ones, and few)
    IH, IW = 11, 7
    OH, OW, pt, pl = ops.conv2d_geometry(IH, IW, FH, FW, covered, sy, sx, dy, dx)
    B = 3 if many == 0 else -(-50000 * 16 // (OH * OW * FH * FW * C * np.dtype(dtype).itemsize)) + 1
    r = rng(FH * 100 + FW * 10 + C)
    im = nrm(r, (B, IH, IW, C)).astype(dtype)
    want = oracle_port.im2col(f(im), OH, OW, FH, FW, sy, sx, dy, dx, pt, pl).astype(dtype).ravel()
    di, dc = DeviceArray.from_numpy(im), DeviceArray.from_numpy(np.full(before + want.size + 32, 7, dtype))
    check(lib.d8_im2col(capi.FLOAT16 if dtype == np.float16 else capi.FLOAT32, di.ptr, dc.ptr + before * im.itemsize, B, IH, IW, C, OH, OW, FH, FW, sy, sx, dy, dx, pt, pl, None))
    got, bits = dc.numpy(), np.uint16 if dtype == np.float16 else np.uint32
    assert np.array_equal(got[before:before + want.size].view(bits), want.view(bits))
    assert (got[:before] == 7).all() and (got[before + want.size:] == 7).all()
