"""The launch shape and row indexing that generated kernels are given, read from
their source: how a periodic row's index is formed."""
import pytest

import manifesto_amd as M
import oracle as O

F, B, H = M.FLOAT32, M.BFLOAT16, M.FLOAT16
FULL, ROW = M.OPERAND_FULL, M.OPERAND_PERIODIC


def source(tree, operands, out):
    return M.FusedKernel(O.flatten(tree), operands, out, "shape").source


# rows of whole items take the constant remainder; others the scalar one
@pytest.mark.parametrize("dt, period, scalar", [(B, 14336, False), (H, 768, False), (H, 24, False), (F, 12, False),
                                                (B, 2730, True), (H, 12, True), (F, 7, True), (B, 4, False)])
def test_row_index(dt, period, scalar):
    src = source((O.N_ADD, ("in", 0), ("in", 1)), [(dt, FULL, 0), (dt, ROW, period)], dt)
    loop = src.split("EmitHIP")[1]
    assert (f"mfh_row_index<{period}ull>(e0)" in loop) == scalar
    assert (f"(e0 % {period}LL)" in loop) == (not scalar)
