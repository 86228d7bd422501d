"""GPU parity of the Int4 dequant over every kind of group size: multiples of
an item's elements and not (an item then reads two scales), below and above
2^15 (the two forms of the group number) and 2^16, groups that end at an
item's first and last element, and scales that are not finite, to the bit."""
import numpy as np
import pytest

import manifesto_amd as M
import oracle as O

from test_gpu_dequant import int4_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    M.init(0)


@pytest.mark.parametrize("group", [4, 5, 8, 9, 12, 15, 17, 96, 100, 1001, 4094, 14336, 32760, 32767, 32768, 32769, 40000,
                                   65528, 65535, 65536, 65537, 100001])
@pytest.mark.parametrize("scale_dt, out_dt", [(O.FLOAT32, O.BFLOAT16), (O.FLOAT16, O.FLOAT32), (O.BFLOAT16, O.FLOAT16)])
def test_any_group_size(group, scale_dt, out_dt):
    rng = np.random.default_rng(group + scale_dt)
    n = max(3 * group + 13, 3 * 16384 + 13)  # several chunks and groups, partial last ones, odd
    int4_case(n, group, scale_dt, out_dt, rng.uniform(-0.05, 0.05, n // group + 2).astype(np.float32), rng, pad=group % 2)


@pytest.mark.parametrize("group", [9, 100, 40001])
def test_split_items_with_scales_that_are_not_finite(group):
    rng = np.random.default_rng(group)
    n = 5 * max(group, 8192) + 3
    scales = np.resize(np.array([0.01, np.inf, -0.02, np.nan, -np.inf, 0.0, 1e30, -0.0], np.float32), n // group + 2)
    for out_dt in (O.BFLOAT16, O.FLOAT32):
        int4_case(n, group, O.FLOAT32, out_dt, scales, rng)


# pad 1 puts a 16-bit output off its dwords, which runs the default shape
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("items, threads", [(1, 64), (2, 128), (4, 512)])
def test_launch_shapes(items, threads, pad):
    rng = np.random.default_rng(items)
    try:
        M.set_launch_config("int4", 0, items)
        M.set_launch_threads("int4", threads)
        for group in (64, 100, 40001):
            n = 5 * 16384 + 7
            int4_case(n, group, O.FLOAT16, O.BFLOAT16, rng.uniform(0.005, 0.02, n // group + 2).astype(np.float32), rng, pad)
    finally:
        M.set_launch_config("int4", -1, -1)
        M.set_launch_threads("int4", -1)
