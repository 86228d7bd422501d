"""Chains that the device compiler could not translate compile.  Each runs in a
process of its own: such a failure aborts the process."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
sys.path.insert(0, {root!r})
import manifesto_amd as M
import oracle as O
flags = M.FUSION_PRECISE | M.FUSION_NO_ROUNDING_TEST
M.FusedKernel(O.flatten((O.N_TANH, ("in", 0))), [({dt}, M.OPERAND_FULL, 0)], {out}, "tanh", flags).close()
print("compiled")
"""


@pytest.mark.parametrize("dt, out", [("M.FLOAT16", "M.BFLOAT16"), ("M.BFLOAT16", "M.FLOAT16"), ("M.FLOAT16", "M.FLOAT16")])
def test_reference_tanh_between_16_bit_types(dt, out, tmp_path):
    # the library's f64 tanh ends in a copysign that was carried through both
    # conversions; the disk cache of compiled kernels is a fresh one
    env = dict(os.environ, MFH_KERNEL_CACHE_DIR=str(tmp_path))
    r = subprocess.run([sys.executable, "-c", CHILD.format(root=ROOT, dt=dt, out=out)], env=env, capture_output=True, text=True)
    assert r.returncode == 0 and "compiled" in r.stdout, r.stderr[:400]
