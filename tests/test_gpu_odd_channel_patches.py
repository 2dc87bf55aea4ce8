"""Conv2d of channel counts that no 16-byte piece divides: patch rows whose pieces cross taps, rows of the filter and their own end; padding
and strides on every side.  Integers against the oracle, bit for bit."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("FH,FW,sy,sx,dy,dx", [(1, 1, 1, 1, 1, 1), (1, 4, 1, 2, 1, 1), (3, 1, 2, 1, 1, 1), (3, 3, 1, 1, 1, 1), (3, 3, 2, 2, 1, 1), (5, 4, 1, 1, 1, 2), (2, 7, 3, 1, 2, 1)])
@pytest.mark.parametrize("IC,OC", [(5, 64), (7, 33), (13, 72), (29, 16), (134, 40)])
@pytest.mark.parametrize("covered", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_forward_and_filter_gradient(oracle_port, FH, FW, sy, sx, dy, dx, IC, OC, covered, dtype):
    from deep8_amd import ops
    B, IH, IW, geo = 3, 15, 14, (covered, sy, sx, dy, dx)
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(FH * 100 + FW * 10 + IC)
    x, w = ints(r, (B, IH, IW, IC), 2) * (r.random((B, IH, IW, IC)) < 0.4), ints(r, (OC, FH, FW, IC), 2) * (r.random((OC, FH, FW, IC)) < 0.4)
    gz = ints(r, (B, OH, OW, OC), 2) * (r.random((B, OH, OW, OC)) < 0.4)
    z, gw = oracle_port.conv2d(x, w, *geo), oracle_port.conv2d_grad_y(x, w, gz, *geo)
    assert max(np.abs(z).max(), np.abs(gw).max()) < 2000
    x, w, gz = (a.astype(dtype) for a in (x, w, gz))
    assert np.array_equal(f(ops.conv2d(x, w, *geo)), z)
    assert np.array_equal(f(ops.conv2d_grad_y(x, w, gz, *geo)), gw)
