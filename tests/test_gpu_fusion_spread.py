"""Kernels of two items per thread around the launch size from which a thread
takes its second item: the same bits as with one item per thread, nothing
written past the output."""
import numpy as np
import pytest

import manifesto_amd as M
import oracle as O

from gpu_util import empty_dev, stream, to_dev, to_host

pytestmark = pytest.mark.gpu

SIZE = {O.FLOAT32: 4, O.BFLOAT16: 2}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    M.init(0)


@pytest.mark.parametrize("dt, operands, vec", [(O.FLOAT32, 1, 4), (O.BFLOAT16, 1, 8), (O.BFLOAT16, 2, 8)])
def test_threads_take_one_item_or_two(dt, operands, vec):
    import torch
    compute_units = torch.cuda.get_device_properties(0).multi_processor_count
    limit = compute_units * 4 * 2 * 64  # items
    tree = (O.N_SIGMOID, ("in", 0)) if operands == 1 else (O.N_MUL, (O.N_SIGMOID, ("in", 0)), ("in", 1))
    ops = [(dt, M.OPERAND_FULL, 0)] * operands
    two = M.FusedKernel(O.flatten(tree), ops, dt, "two")
    assert f"{vec} elements per item, 2 item(s) per thread" in two.source
    try:
        M.set_launch_config("fused", 0, 1)
        one = M.FusedKernel(O.flatten(tree), ops, dt, "one")
    finally:
        M.set_launch_config("fused", -1, -1)
    rng = np.random.default_rng(limit + vec)
    top = (limit + 2) * vec
    devs = [to_dev(O.encode(rng.normal(0, 2, top).astype(np.float32), dt)) for _ in range(operands)]
    for count in (1, vec, 64 * vec + 1, limit * vec - 1, limit * vec, limit * vec + vec - 1, (limit + 1) * vec, top):
        got = []
        for k in (two, one):
            out, op = empty_dev(count * SIZE[dt] + 64)
            k.launch([p for _, p in devs], op, count, stream())
            got.append(to_host(out, np.uint8))
            assert (got[-1][count * SIZE[dt]:] == 0xA5).all(), f"count {count}: wrote past the output"
        assert np.array_equal(*got), f"count {count}"
