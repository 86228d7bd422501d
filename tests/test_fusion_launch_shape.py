"""The launch shape and row indexing that generated kernels are given, read from
their source: how many items a thread takes by the widths of the streams, and
how a periodic row's index is formed."""
import pytest

import manifesto_amd as M
import oracle as O

F, B, H = M.FLOAT32, M.BFLOAT16, M.FLOAT16
FULL, ROW = M.OPERAND_FULL, M.OPERAND_PERIODIC


def source(tree, operands, out):
    return M.FusedKernel(O.flatten(tree), operands, out, "shape").source


def product(node, operands, out):
    tree = (O.N_MUL, (node, ("in", 0)), ("in", 1))
    for k in range(2, len(operands)):
        tree = (O.N_ADD, tree, ("in", k))
    return source(tree, operands, out)


def full(*dts):
    return [(dt, FULL, 0) for dt in dts]


@pytest.mark.parametrize("node", [O.N_SIGMOID, O.N_SILU, O.N_TANH, O.N_GELU])
@pytest.mark.parametrize("operands, out, items", [
    (full(F, F), F, 1), (full(F, F), B, 1), (full(F, F, F), F, 1), (full(B, B), F, 1), (full(F, H), F, 1),
    # few bytes in flight per item
    (full(F, B), B, 2), (full(H, F), H, 2), (full(B, B) + [(F, ROW, 4096)], B, 2)])
def test_items_per_thread_of_two_operands(node, operands, out, items):
    if node == O.N_GELU and out == F and operands[0][0] != operands[1][0]:
        items = 2
    assert f"4 elements per item, {items} item(s) per thread" in product(node, operands, out)


@pytest.mark.parametrize("node", [O.N_SIGMOID, O.N_LOG, O.N_TANH])
@pytest.mark.parametrize("dt, out", [(F, F), (F, B), (B, F)])
def test_items_per_thread_of_one_operand(node, dt, out):
    assert "4 elements per item, 2 item(s) per thread" in source((node, ("in", 0)), full(dt), out)


@pytest.mark.parametrize("node, operands, out", [
    (O.N_LOG, full(F, B), B), (O.N_LOG, full(B, B) + [(F, ROW, 4096)], B),
    (O.N_EXP, full(F, B), B), (O.N_EXP, full(F, F), F), (O.N_EXP, full(B, B), B)])
def test_two_operands_of_a_log_or_an_exp_take_one_item(node, operands, out):
    assert "elements per item, 1 item(s) per thread" in product(node, operands, out)


# rows of whole items take the constant remainder; others the scalar one
@pytest.mark.parametrize("dt, period, scalar", [(B, 14336, False), (H, 768, False), (H, 24, False), (F, 12, False),
                                                (B, 2730, True), (H, 12, True), (F, 7, True), (B, 4, False)])
def test_row_index(dt, period, scalar):
    src = source((O.N_ADD, ("in", 0), ("in", 1)), [(dt, FULL, 0), (dt, ROW, period)], dt)
    loop = src.split("EmitHIP")[1]
    assert (f"mfh_row_index<{period}ull>(e0)" in loop) == scalar
    assert (f"(e0 % {period}LL)" in loop) == (not scalar)
