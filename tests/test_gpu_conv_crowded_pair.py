"""Both gradients of an fp32 convolution in one launch of more workgroups than run at once: on either side of the line that the length of a
workgroup draws, with a cut K step, in pieces or not.  One call leaves the bits of two calls, which their own tests hold to the oracle."""
import numpy as np
import pytest

from util import nrm, rng

pytestmark = pytest.mark.gpu


# B, IH, IW, IC, OC, F, covered, stride, dilation; whether the two share a launch for being crowded
@pytest.mark.parametrize("cfg,crowded", [((3, 79, 79, 48, 64, 3, 1, 1, 1), 1), ((7, 35, 35, 64, 64, 5, 0, 1, 2), 1), ((17, 17, 17, 200, 148, 3, 1, 1, 1), 1),
                                         ((13, 25, 25, 192, 64, 3, 0, 1, 1), 1), ((29, 75, 75, 64, 32, 1, 1, 1, 1), 1), ((4, 82, 82, 64, 168, 3, 1, 1, 1), 0)])
def test_one_call_leaves_what_two_leave(cfg, crowded):
    from deep8_amd import capi, ops
    lib = capi.init()
    B, IH, IW, IC, OC, F, covered, stride, dilation = cfg
    geo = (bool(covered), stride, stride, dilation, dilation)
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, F, F, *geo)
    r = rng(sum(cfg))
    x, w, gz = (nrm(r, s).astype(np.float32) for s in ((B, IH, IW, IC), (OC, F, F, IC), (B, OH, OW, OC)))
    gx0, gw0 = nrm(r, x.shape).astype(np.float32), nrm(r, w.shape).astype(np.float32)
    before = lib.d8_conv_grad_crowded_pair_launches()
    gx, gw = ops.conv2d_grad_xy(x, w, gz, *geo, gx=gx0, gw=gw0, overwrite_w=True)
    assert lib.d8_conv_grad_crowded_pair_launches() - before == crowded
    assert np.array_equal(gx.view(np.uint32), ops.conv2d_grad_x(x, w, gz, *geo, gx=gx0).view(np.uint32))
    assert np.array_equal(gw.view(np.uint32), ops.conv2d_grad_y(x, w, gz, *geo, overwrite=True).view(np.uint32))
