"""GPU parity of fused chains where whole items and rows do not line up: a
periodic row of any length (shorter than an item, not a multiple of one,
ending inside one) and buffers aligned to their element only.  The chain is
arithmetic, so every result is the oracle's to the bit."""
import numpy as np
import pytest

import manifesto_amd as M
import oracle as O

from test_gpu_fusion import run_fused

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    M.init(0)


# (x + row) * s + r: the row is an Add operand (an f16 pair takes the packed
# form), and again alone
CHAIN = O.flatten((O.N_ADD, (O.N_MUL, (O.N_ADD, ("in", 0), ("in", 1)), ("in", 2)), ("in", 3)))


@pytest.mark.parametrize("dt", [O.FLOAT32, O.BFLOAT16, O.FLOAT16])
@pytest.mark.parametrize("period", [1, 3, 7, 8, 9, 12, 24, 511, 2730, 14336])
@pytest.mark.parametrize("pads", [(0, 0, 0), (1, 0, 3), (3, 5, 1)])
def test_any_row_length_and_element_alignment(dt, period, pads):
    count = max(3 * period + 5, 2 * 64 * 8 * 3 + 5)  # ragged last row, several waves
    rng = np.random.default_rng(period * 7 + dt + sum(pads))
    x, r = (O.encode(rng.normal(0, 2, count).astype(np.float32), dt) for _ in range(2))
    row = O.encode(rng.normal(0, 2, period).astype(np.float32), dt)
    s = np.array([1.375], np.float32)
    ops = [(dt, M.OPERAND_FULL, 0), (dt, M.OPERAND_PERIODIC, period), (O.FLOAT32, M.OPERAND_SCALAR, 0),
           (dt, M.OPERAND_FULL, 0)]
    # run_fused gives the output the first input's offset
    got = run_fused(CHAIN, ops, [x, row, s, r], dt, count, pads=[pads[0], pads[1], 0, pads[2]], name="ragged")
    ins = [O.decode(x, dt), O.decode(row, dt), s, O.decode(r, dt)]
    want = O.encode(O.run(CHAIN, ins, count, periods=[0, period, 1, 0]), dt)
    bad = np.flatnonzero(got.view(np.uint8) != want.view(np.uint8))
    assert bad.size == 0, f"dt={dt} period={period} pads={pads}: first difference at byte {bad[0]}"


@pytest.mark.parametrize("period", [5, 6, 4095])
def test_mixed_dtypes_with_rows_of_two_lengths(period):
    # f32 in, bf16 and f16 rows: items of four elements; both rows end inside items
    n = 4 * 64 * 6 + 3
    rng = np.random.default_rng(period)
    x = rng.normal(0, 2, n).astype(np.float32)
    a = O.encode(rng.normal(0, 1, period).astype(np.float32), O.BFLOAT16)
    b = O.encode(rng.normal(0, 1, 10).astype(np.float32), O.FLOAT16)
    nodes = O.flatten((O.N_SUB, (O.N_MUL, ("in", 0), ("in", 1)), ("in", 2)))
    ops = [(O.FLOAT32, M.OPERAND_FULL, 0), (O.BFLOAT16, M.OPERAND_PERIODIC, period),
           (O.FLOAT16, M.OPERAND_PERIODIC, 10)]
    got = run_fused(nodes, ops, [x, a, b], O.FLOAT32, n, pads=[1, 1, 1], name="rows2")
    want = O.run(nodes, [x, O.decode(a, O.BFLOAT16), O.decode(b, O.FLOAT16)], n, periods=[0, period, 10])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
