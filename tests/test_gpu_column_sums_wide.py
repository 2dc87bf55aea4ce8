"""Column sums of few rows in one launch: columns on both sides of the lines between 4, 8 and 32 threads across (512 and 4096 pieces
of 16 bytes).  Integers, so every order of additions gives the same."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [65, 128, 129, 512])
@pytest.mark.parametrize("pieces", [511, 512, 513, 4095, 4096, 4097, 4130])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_columns_around_the_lines(rows, pieces, dtype):
    from deep8_amd import ops
    cols = pieces * 16 // np.dtype(dtype).itemsize
    r = rng(rows * 5000 + pieces)
    dz = r.integers(-2, 3, (rows, cols), dtype=np.int8).astype(dtype)
    g = ints(r, (cols,), 3).astype(dtype)
    sums = dz.astype(np.float32).sum(axis=0)
    got = ops.add_grad(g.reshape(1, 1, cols), dz.reshape(1, rows, cols))
    assert np.array_equal(got.reshape(cols), (sums + g).astype(dtype))
    z = r.integers(-1, 2, (rows, cols), dtype=np.int8).astype(dtype)
    gated = np.where(z > 0, dz, 0).astype(dtype)
    dpre, db = ops.bias_relu_grad(z, dz, g, True, False)
    assert np.array_equal(dpre, gated)
    assert np.array_equal(db, (gated.astype(np.float32).sum(axis=0) + g).astype(dtype))
