"""d8_bias_relu_grad on rows that start at any element (an odd number of columns, an element-aligned tensor): 16-byte
accesses whose last one in a row shares columns with its neighbour.  Integers against numpy, so everything is exact
(sums stay below 2048, where Float16 counts in ones); reals bit for bit against ReLuGrad followed by AddGrad."""
import numpy as np
import pytest

from util import ints, nrm, rng

pytestmark = pytest.mark.gpu

# columns at the ends of the rule (more than 16 pieces of 16 bytes: 65 / 129), one past / one short of whole pieces, more than
# one column group (256 / 128), rows that are no multiple of the row lanes or of the chunks, a single row
SHAPES = [(1, 1001), (7, 65), (64, 129), (65, 130), (130, 135), (257, 137), (1000, 257), (513, 1001), (5000, 131), (31, 2047)]


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("in_place", [False, True])
def test_gate_any_columns(rows, cols, dtype, in_place):
    from deep8_amd import ops
    r = rng(rows + cols)
    z = np.maximum(nrm(r, (rows, cols)), 0).astype(dtype)
    dz = ((ints(r, (rows, cols), 3) - 1) * (r.random((rows, cols)) < min(1.0, 600.0 / rows))).astype(dtype)
    want = np.where(z > 0, dz, 0).astype(dtype)
    sums = want.astype(np.float64).sum(axis=0)
    assert np.abs(sums).max() < 2040
    db0 = ints(r, (cols,), 5).astype(dtype)
    for use_scratch in (True, False):
        dpre, db = ops.bias_relu_grad(z, dz, db0, use_scratch, in_place)
        assert np.array_equal(dpre, want) and np.array_equal(db, (sums + db0).astype(dtype)), use_scratch
        dpre, db = ops.bias_relu_grad(z, dz, None, use_scratch, in_place)  # written over NaN
        assert np.array_equal(dpre, want) and np.array_equal(db, sums.astype(dtype)), use_scratch
    reals = nrm(r, (rows, cols)).astype(dtype)
    dpre, db = ops.bias_relu_grad(z, reals, np.zeros(cols, dtype), True, in_place)
    seq = ops.relu_grad(z, reals, overwrite=True)
    assert np.array_equal(dpre, seq)
    seq_db = ops.add_grad(np.zeros((1, cols), dtype), seq.reshape(1, rows, cols) if rows > 1 else seq)
    assert np.array_equal(db, seq_db.reshape(cols))


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("cols", [256, 131])
def test_gate_element_aligned_tensors(dtype, cols):
    """tensors that start one element into a block, with guards around what is written"""
    from deep8_amd import capi
    lib = capi.init()
    rows, r = 130, rng(cols)
    z = np.maximum(nrm(r, (rows, cols)), 0).astype(dtype)
    dz = (ints(r, (rows, cols), 3) - 1).astype(dtype)
    pad = lambda v: np.concatenate([np.full(1, 7, dtype), v.ravel(), np.full(9, 7, dtype)])
    dev = [capi.DeviceArray.from_numpy(pad(v)) for v in (z, dz, np.zeros_like(dz), np.zeros(cols, dtype))]
    at = [d.ptr + z.itemsize for d in dev]
    dt = capi.FLOAT32 if dtype == np.float32 else capi.FLOAT16
    capi.check(lib.d8_bias_relu_grad(dt, *at, rows, cols, 0, None, 0, None))
    want = np.where(z > 0, dz, 0).astype(dtype)
    assert np.array_equal(dev[2].numpy(), pad(want))
    assert np.array_equal(dev[3].numpy(), pad(want.astype(np.float64).sum(axis=0).astype(dtype)))
