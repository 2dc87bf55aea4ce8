"""Conv2d forward and filter gradient on images of few channels, which are read from LDS instead of through a patch matrix
(D8_CONV_DIRECT: also where the matrix is expected to be faster): whole numbers bit for bit against the oracle, an infinity in the
image (what fills a run or a row up must not meet it), and tensors that start at any element."""
import numpy as np
import pytest

from util import f, h, ints, rng

pytestmark = pytest.mark.gpu

# B, IH, IW, IC, OC, FH, FW, covered, sy, sx, dy, dx
CASES = [
    (2, 28, 28, 1, 32, 5, 5, True, 1, 1, 1, 1),     # one block of channels, one of the gradient's columns
    (1, 30, 31, 3, 64, 7, 7, True, 2, 2, 1, 1),     # rows of odd length; the longest patch row, five blocks of columns
    (2, 32, 48, 3, 64, 7, 7, True, 2, 2, 1, 1),     # ... rows that move in 16-byte pieces
    (2, 17, 23, 3, 40, 3, 3, False, 1, 1, 1, 1),    # channels that end inside a block
    (1, 9, 300, 1, 8, 3, 3, True, 1, 1, 1, 1),      # a row of several tiles
    (3, 5, 4, 3, 72, 3, 3, True, 1, 1, 2, 1),       # a dilation along y, an image smaller than the filter's reach
    (2, 16, 16, 5, 17, 1, 1, True, 1, 1, 1, 1),     # one tap, channels that cannot be moved in pieces
    (1, 40, 36, 2, 96, 5, 5, True, 2, 1, 1, 1),     # two groups of output channels
    (2, 13, 13, 1, 130, 7, 7, True, 1, 2, 1, 1),
    (600, 6, 8, 1, 8, 3, 3, True, 1, 1, 1, 1),      # more tiles than workgroups
    (3, 20, 20, 3, 192, 3, 3, True, 2, 2, 1, 1),    # whole groups of 64 output channels
    (3, 20, 20, 3, 193, 3, 3, True, 2, 2, 2, 1),    # ... and one channel more; the image rows two apart
    (2, 9, 9, 3, 321, 5, 5, True, 1, 1, 1, 1),      # six groups
    (2, 12, 12, 6, 24, 3, 4, False, 1, 3, 1, 1),
]


def _shifted(a, elements):
    """a tensor that starts `elements` elements into its allocation"""
    from deep8_amd.capi import DeviceArray
    flat = np.concatenate([np.full(elements, np.nan, a.dtype), a.ravel(), np.full(8, np.nan, a.dtype)])
    d = DeviceArray.from_numpy(flat)
    return d, d.ptr + elements * a.itemsize


@pytest.mark.parametrize("cfg", CASES)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("start,infinite", [(0, False), (1, False), (0, True)])
def test_few_channels(oracle_port, cfg, dtype, start, infinite, monkeypatch):
    monkeypatch.setenv("D8_CONV_DIRECT", "1")
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = ops.conv2d_geometry(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]))
    hi = 3 if dtype == np.float16 else 10
    c = (lambda v: h(v)) if dtype == np.float16 else (lambda v: v)
    x, w, gz = ints(r, (B, IH, IW, IC), hi), ints(r, (OC, FH, FW, IC), hi), ints(r, (B, OH, OW, OC), hi)
    old, bias = ints(r, w.shape, hi), ints(r, (OC,), hi)
    gz = gz * (r.random(gz.shape) < min(1.0, 300.0 / (B * OH * OW)))  # thinned: sums that half holds
    if infinite:
        x[B // 2, IH // 2, IW // 2, 0] = np.inf
    z = oracle_port.conv2d(x, w, *geo)
    want_z = np.maximum(z + bias, 0) if not infinite else z
    want_gw = oracle_port.conv2d_grad_y(x, w, gz, *geo)
    fin = lambda t: np.abs(t[np.isfinite(t)]).max(initial=0.0)
    assert dtype == np.float32 or max(fin(want_z), fin(want_gw)) < 2040
    dt, es = capi.dtype_id(np.dtype(dtype)), np.dtype(dtype).itemsize
    shape, filt, g = (B, IH, IW, IC), (OC, FH, FW), (int(geo[0]),) + tuple(geo[1:])
    (dx, px), (dw, pw), (dg, pg), (db, pb) = (_shifted(c(t), start) for t in (x, w, gz, bias))
    nan = lambda shape: np.full(shape, np.nan, dtype)
    need = [lib.d8_conv2d_scratch_bytes(dt, k, *shape, *filt, *g) for k in (0, 2)]
    ws = DeviceArray((max(need),), np.uint8)
    before = lib.d8_conv_route_calls(2)
    out, po = _shifted(nan(want_z.shape), start)
    if infinite:
        check(lib.d8_conv2d(dt, px, *shape, pw, *filt, po, *g, ws.ptr, need[0], None))
    else:
        check(lib.d8_conv2d_bias_relu(dt, px, *shape, pw, *filt, pb, 1, po, *g, ws.ptr, need[0], None))
    got = f(out.numpy())
    n = want_z.size
    assert np.array_equal(got[start:start + n].reshape(want_z.shape), want_z, equal_nan=True)
    assert np.isnan(got[:start]).all() and np.isnan(got[start + n:]).all()
    n = want_gw.size
    for name, there, want in (("d8_conv2d_grad_y_overwrite", nan(w.shape), want_gw), ("d8_conv2d_grad_y", c(old), want_gw + old)):
        out, po = _shifted(there, start)
        check(getattr(lib, name)(dt, px, *shape, po, *filt, pg, *g, ws.ptr, need[1], None))
        got = f(out.numpy())
        assert np.array_equal(got[start:start + n].reshape(w.shape), want, equal_nan=True), name
        assert np.isnan(got[:start]).all() and np.isnan(got[start + n:]).all()
    assert lib.d8_conv_route_calls(2) == before + 3


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_more_groups_of_channels_than_a_grid_takes(dtype, monkeypatch):
    """groups of 32 output channels beyond the grid's second dimension: the layer keeps the patch matrix"""
    monkeypatch.setenv("D8_CONV_DIRECT", "1")
    from deep8_amd import capi, ops
    lib = capi.init()
    OC = 65536 * 32
    r = rng(7)
    x, w = ints(r, (1, 4, 4, 1), 3), r.integers(0, 3, size=(OC, 3, 3, 1), dtype=np.int8)
    gz = np.zeros((1, 2, 2, OC), dtype)
    gz[0, 1, 0, ::1000] = 1
    patches = np.stack([x[0, i:i + 3, j:j + 3, 0].ravel() for i in range(2) for j in range(2)])
    before = lib.d8_conv_route_calls(0), lib.d8_conv_route_calls(2)
    z = ops.conv2d(x.astype(dtype), w.astype(dtype), False)
    assert np.array_equal(z.reshape(4, OC), (patches @ w.reshape(OC, 9).T.astype(np.float32)).astype(dtype))
    gw = ops.conv2d_grad_y(x.astype(dtype), w.astype(dtype), gz, False)
    assert np.array_equal(gw.reshape(OC, 9), gz[0, 1, 0][:, None] * patches[2].astype(dtype))
    assert (lib.d8_conv_route_calls(0), lib.d8_conv_route_calls(2)) == (before[0] + 2, before[1])
