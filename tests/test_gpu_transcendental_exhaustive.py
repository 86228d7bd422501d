"""Every f32 input through the device's Exp, Log and Tanh nodes and through
divisions by a constant: the rounding-tested forms must give the bit patterns
of the reference forms evaluated on every element
(MFH_FUSION_NO_ROUNDING_TEST; codegen/cpu.go:150-185), NaN positions
included, in chains that stream f32 and, rounded to storage, in 16-bit ones."""
import numpy as np
import pytest

import manifesto_amd as M
import oracle as O

from gpu_util import log, stream

pytestmark = pytest.mark.gpu

CHUNK = 1 << 28
PLAIN = M.FUSION_PRECISE | M.FUSION_NO_ROUNDING_TEST


@pytest.fixture(scope="module", autouse=True)
def gpu():
    M.init(0)


def same_over_every_input(tree, name):
    import torch
    nodes, ops = O.flatten(tree), [(M.FLOAT32, M.OPERAND_FULL, 0)]
    tested = M.FusedKernel(nodes, ops, M.FLOAT32, f"t_{name}")
    plain = M.FusedKernel(nodes, ops, M.FLOAT32, f"p_{name}", PLAIN)
    a = torch.empty(CHUNK, dtype=torch.int32, device="cuda")
    b = torch.empty(CHUNK, dtype=torch.int32, device="cuda")
    for c in range((1 << 32) // CHUNK):
        x = (torch.arange(c * CHUNK, (c + 1) * CHUNK, dtype=torch.int64, device="cuda") - (1 << 31)).to(torch.int32)
        tested.launch([x.data_ptr()], a.data_ptr(), CHUNK, stream())
        plain.launch([x.data_ptr()], b.data_ptr(), CHUNK, stream())
        nan_a, nan_b = (a & 0x7FFFFFFF) > 0x7F800000, (b & 0x7FFFFFFF) > 0x7F800000
        idx = torch.nonzero((nan_a != nan_b) | ((a != b) & ~nan_b)).flatten()
        if idx.numel():
            i = idx[:4].cpu().tolist()
            raise AssertionError(f"{name}: {idx.numel()} inputs differ in chunk {c}, e.g. x bits "
                                 f"{[hex(int(x[j]) & 0xFFFFFFFF) for j in i]}: tested {[hex(int(a[j]) & 0xFFFFFFFF) for j in i]}"
                                 f" plain {[hex(int(b[j]) & 0xFFFFFFFF) for j in i]}")
    log(f"{name}: every f32 input identical")


@pytest.mark.parametrize("node", [O.N_EXP, O.N_LOG, O.N_TANH])
def test_every_f32_input(node):
    same_over_every_input((node, ("in", 0)), f"node_{node}")


# 6: quotients that are subnormal ties; 1e-40: a subnormal divisor; 2^-3: exact
@pytest.mark.parametrize("c", [30.0, 3.0, 6.0, -1.1, 0.125, 0.0070000002, 1.9999998807907104, 1e30, 1e-40])
def test_division_by_a_constant(c):
    # x / c + e^-200 (= 0): the chain holds a transcendental node, so the
    # division takes the reciprocal form
    tree = (O.N_ADD, (O.N_DIV, ("in", 0), ("const", c)), (O.N_EXP, ("const", -200.0)))
    src = M.FusedKernel(O.flatten(tree), [(M.FLOAT32, M.OPERAND_FULL, 0)], M.FLOAT32, "d").source
    assert "mfh_div_const(x0" in src
    same_over_every_input(tree, f"div_{c}")


@pytest.mark.parametrize("dt", [O.BFLOAT16, O.FLOAT16])
@pytest.mark.parametrize("node", [O.N_EXP, O.N_LOG, O.N_TANH])
def test_every_16bit_code(node, dt):
    # the element loop too: an odd count leaves a tail
    import torch
    codes = torch.arange(-32768, 32768, dtype=torch.int32, device="cuda").to(torch.int16).repeat(3)[:-1].contiguous()
    outs = []
    for flags in (0, PLAIN):
        k = M.FusedKernel(O.flatten((node, ("in", 0))), [(dt, M.OPERAND_FULL, 0)], dt, "c", flags)
        out = torch.empty_like(codes)
        k.launch([codes.data_ptr()], out.data_ptr(), codes.numel(), stream())
        outs.append(out)
    limit = 0x7F80 if dt == O.BFLOAT16 else 0x7C00
    nan = [(o & 0x7FFF) > limit for o in outs]
    assert torch.equal(nan[0], nan[1])
    assert torch.equal(outs[0][~nan[0]], outs[1][~nan[0]])


def test_masked_and_special_values():
    # e^v of a masked score (the lowest value of the type, -Inf) is 0; zeros,
    # infinities and ones through each node
    v = np.array([-3.4028235e38, -np.inf, np.inf, 0.0, -0.0, 1.0, 2.0 ** -126, -200.0, 100.0], np.float32)
    import torch
    x = torch.from_numpy(np.resize(v, 4096)).cuda()
    for node in (O.N_EXP, O.N_LOG, O.N_TANH):
        out = torch.empty_like(x)
        M.FusedKernel(O.flatten((node, ("in", 0))), [(M.FLOAT32, 0, 0)], M.FLOAT32, "m").launch(
            [x.data_ptr()], out.data_ptr(), 4096, stream())
        got, want = out.cpu().numpy(), O.eval_unary(node, np.resize(v, 4096))
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
