"""Column sums of few rows, where a launch of narrow blocks takes the place of chunks and a second launch: the row counts on both
sides of its lines, columns that leave the last block's vectors unused, and columns (half 4, 268) that keep the chunks.  Integers,
so every order of additions gives the same."""
import numpy as np
import pytest

from util import ints, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [64, 65, 127, 128, 129, 511, 512, 513])
@pytest.mark.parametrize("cols", [4, 8, 40, 264, 268, 1032])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_rows_around_the_lines(rows, cols, dtype):
    from deep8_amd import ops
    r = rng(rows * 2000 + cols)
    dz = ints(r, (rows, cols), 2).astype(dtype)
    g = ints(r, (cols,), 3).astype(dtype)
    sums = dz.astype(np.float64).sum(axis=0)
    assert np.abs(sums).max() < 2040
    got = ops.add_grad(g.reshape(1, 1, cols), dz.reshape(1, rows, cols))
    assert np.array_equal(got.reshape(cols), (sums + g).astype(dtype))
    z = ints(r, (rows, cols), 2).astype(dtype)
    gated = np.where(z > 0, dz, 0).astype(dtype)
    dpre, db = ops.bias_relu_grad(z, dz, g, True, False)
    assert np.array_equal(dpre, gated)
    assert np.array_equal(db, (gated.astype(np.float64).sum(axis=0) + g).astype(dtype))
