"""What the scratch queries of a half MatrixMultiply with odd rows ask for: room for a copy of each operand, also where the two have
one shape (they are still two matrices)."""
import pytest


def _copy(rows, cols):
    return rows * ((cols + 63) // 64 * 64) * 2


@pytest.mark.parametrize("xb,R,I,yb,O", [(1, 515, 515, 1, 515), (1, 2001, 2001, 1, 2001), (3, 203, 203, 3, 203), (1, 515, 515, 1, 517), (2, 515, 131, 1, 645)])
def test_forward_copies_of_both_operands(monkeypatch, xb, R, I, yb, O):
    from deep8_amd import capi
    lib = capi.load()
    monkeypatch.setenv("D8_GEMM_PACK", "0")
    plain = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 0, xb, R, I, yb, I, O)
    monkeypatch.setenv("D8_GEMM_PACK", "1")
    asked = lib.d8_matmul_scratch_bytes(capi.FLOAT16, 0, xb, R, I, yb, I, O)
    assert asked - plain == _copy(xb * R, I) + _copy(yb * I, O)
