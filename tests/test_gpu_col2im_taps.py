"""col2im and the gradient that writes instead of adding: numbers of taps on both sides of multiples of five, strides that leave pixels
without a tap, channels that are moved one by one and in whole pieces.  fp32 bit for bit against the oracle, half on integers."""
import numpy as np
import pytest

from util import f, ints, nrm, rng

pytestmark = pytest.mark.gpu

FILTERS = [(1, 1, 1, 1, 1, 1), (1, 4, 1, 1, 1, 1), (5, 1, 1, 1, 1, 1), (2, 3, 1, 2, 1, 1), (3, 3, 1, 1, 1, 1), (3, 3, 2, 2, 1, 1), (2, 5, 3, 1, 1, 2), (3, 3, 4, 4, 1, 1),
           (3, 4, 1, 1, 2, 1), (7, 7, 2, 2, 1, 1)]


@pytest.mark.parametrize("FH,FW,sy,sx,dy,dx", FILTERS)
@pytest.mark.parametrize("IC", [1, 8, 13, 16])
@pytest.mark.parametrize("covered", [True, False])
def test_taps(oracle_port, FH, FW, sy, sx, dy, dx, IC, covered):
    from deep8_amd import ops
    B, IH, IW = 3, 17, 14
    OH, OW, pt, pl = ops.conv2d_geometry(IH, IW, FH, FW, covered, sy, sx, dy, dx)
    geo = (OH, OW, FH, FW, sy, sx, dy, dx, pt, pl)
    r = rng(FH * 100 + FW * 10 + IC)
    col, im = nrm(r, (B * OH * OW, FH * FW * IC)), nrm(r, (B, IH, IW, IC))
    assert np.array_equal(ops.col2im(col, im, *geo).view(np.uint32), oracle_port.col2im(col, im, *geo).view(np.uint32))
    col, im = ints(r, col.shape, 3).astype(np.float16), ints(r, im.shape, 8).astype(np.float16)
    assert np.array_equal(f(ops.col2im(col, im, *geo)), oracle_port.col2im(f(col), f(im), *geo))


@pytest.mark.parametrize("FH,FW,sy,sx,dy,dx", FILTERS)
@pytest.mark.parametrize("IC,OC", [(13, 40), (70, 33)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_gradient_is_written(oracle_port, FH, FW, sy, sx, dy, dx, IC, OC, dtype):
    from deep8_amd import ops
    B, IH, IW, geo = 2, 15, 12, (True, sy, sx, dy, dx)
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(FH * 100 + FW * 10 + IC)
    x, w, gz = ints(r, (B, IH, IW, IC), 2), ints(r, (OC, FH, FW, IC), 2), ints(r, (B, OH, OW, OC), 2) * (r.random((B, OH, OW, OC)) < 0.3)
    want = oracle_port.conv2d_grad_x(x, w, gz, *geo)
    assert np.abs(want).max() < 2000
    x, w, gz = (a.astype(dtype) for a in (x, w, gz))
    got = ops.conv2d_grad_x(x, w, gz, *geo, gx=np.full(x.shape, np.nan, dtype), overwrite=True)
    assert np.array_equal(f(got), want)
    gx0 = ints(r, x.shape, 2).astype(dtype)
    assert np.array_equal(f(ops.conv2d_grad_x(x, w, gz, *geo, gx=gx0)), want + f(gx0))
