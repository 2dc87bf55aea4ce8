"""Products on the smaller tiles: 64 x 64 where 128-wide tiles would leave compute units idle, 128 x 32 for outputs of at
most 32 columns in fp32; with and without a split reduction, as matrices and as convolutions.  Integers, bit for bit."""
import numpy as np
import pytest

from util import f, ints, rng

pytestmark = pytest.mark.gpu

# M, N, K: either side of a tile, of a band of rows beyond whole rounds of the chip, reductions with and without a rest
SHAPES = [(784, 128, 1152), (130, 191, 608), (65, 260, 999), (1000, 64, 32), (320, 320, 36), (129, 32, 200), (33000, 32, 96),
          (34100, 20, 40), (513, 1, 1000), (128, 31, 2048),
          (384, 512, 700), (384, 513, 700)]  # (either side of where a few pieces are added by a thread per group of outputs)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_products(oracle_port, M, N, K, ta, tb, dtype):
    from deep8_amd import capi
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    r, dt = rng(M + 3 * N + 7 * K), capi.dtype_id(np.dtype(dtype))
    hi = 2 if dtype == np.float16 else 9
    for batch in (1,) if M > 1000 else (1, 3):
        A = ints(r, (batch,) + ((K, M) if ta else (M, K)), hi)
        B = ints(r, (batch,) + ((N, K) if tb else (K, N)), hi)
        C = ints(r, (batch, M, N), 5)
        want = np.stack([oracle_port.gemm(ta, tb, A[i], B[i]) for i in range(batch)])
        assert dtype == np.float32 or want.max() < 2040
        dA, dB = DeviceArray.from_numpy(A.astype(dtype)), DeviceArray.from_numpy(B.astype(dtype))
        asked = lib.d8_gemm_workspace_bytes(dt, ta, tb, M, N, K, batch, M * N)
        for nb, beta in ((asked, 0.0), (asked, 1.0), (0, 0.0), (2 * batch * M * N * 4 + 64, 0.0)):
            dC, ws = DeviceArray.from_numpy(C.astype(dtype)), DeviceArray((max(nb, 16),), np.uint8)
            check(lib.d8_gemm(dt, ta, tb, M, N, K, dA.ptr, A.shape[2], A[0].size, dB.ptr, B.shape[2], B[0].size, beta, dC.ptr, N,
                              M * N, batch, ws.ptr if nb else None, nb, None))
            assert np.array_equal(f(dC.numpy()), want + beta * C), (batch, nb, beta)


# B, IH, IW, IC, OC, FH, FW, covered, sy, sx, dy, dx: few input channels (the gradient of x is narrow), few output channels
CONV = [(2, 28, 28, 32, 64, 5, 5, True, 1, 1, 1, 1), (3, 15, 17, 24, 20, 3, 3, True, 1, 1, 1, 1), (1, 28, 28, 128, 128, 3, 3, True, 1, 1, 1, 1),
        (4, 19, 19, 20, 96, 3, 3, True, 2, 2, 1, 1), (64, 26, 26, 32, 32, 3, 3, False, 1, 1, 1, 1)]
DECONV = [(2, 14, 14, 64, 32, 4, 4, False, 2, 2), (2, 12, 12, 32, 20, 3, 3, False, 1, 1),
          (8, 8, 8, 512, 68, 4, 4, False, 2, 2)]  # (many outputs, stored transposed per tap)


@pytest.mark.parametrize("op,cfg", [("conv2d", c) for c in CONV] + [("deconv2d", c) for c in DECONV])
def test_convolutions(oracle_port, op, cfg):
    from deep8_amd import capi, ops
    from deep8_amd.capi import DeviceArray, check
    lib = capi.init()
    B, IH, IW, IC, OC, FH, FW = cfg[:7]
    geo = cfg[7:]
    OH, OW, _, _ = getattr(ops, op + "_geometry")(IH, IW, FH, FW, *geo)
    r = rng(sum(cfg[:7]))
    x, w, gz = ints(r, (B, IH, IW, IC), 4), ints(r, (OC, FH, FW, IC), 4), ints(r, (B, OH, OW, OC), 4)
    port, g = oracle_port, (int(geo[0]),) + tuple(geo[1:])
    want = [getattr(port, op)(x, w, *geo), getattr(port, op + "_grad_x")(x, w, gz, *geo), getattr(port, op + "_grad_y")(x, w, gz, *geo)]
    for which, name in enumerate(("d8_" + op, "d8_%s_grad_x_overwrite" % op, "d8_%s_grad_y_overwrite" % op)):
        asked = getattr(lib, "d8_%s_scratch_bytes" % op)(capi.FLOAT32, which, B, IH, IW, IC, OC, FH, FW, *g)
        out = DeviceArray.from_numpy(np.full(want[which].shape, np.nan, np.float32))
        bufs = [DeviceArray.from_numpy(t) for t in (x, w, gz)]
        bufs[(2, 0, 1)[which]] = out
        ws = DeviceArray((max(asked, 16),), np.uint8)
        check(getattr(lib, name)(capi.FLOAT32, bufs[0].ptr, B, IH, IW, IC, bufs[1].ptr, OC, FH, FW, bufs[2].ptr, *g, ws.ptr, asked, None))
        assert np.array_equal(out.numpy(), want[which]), name
