"""GPU parity of the ahead-of-time kernels on buffers at any address: whole
items are loaded and stored wherever the buffers stand, so every entry point
runs over several workgroups' chunks and a ragged tail, with the input and the
output each moved off 16 bytes by one element, by an odd number of bytes or by
a dword, and must give the oracle's bytes and touch nothing beside its output."""
import numpy as np
import pytest

import manifesto_amd as M
import oracle as O

from gpu_util import empty_dev, stream, to_dev, to_host

pytestmark = pytest.mark.gpu

SIZE = {O.FLOAT64: 8, O.FLOAT32: 4, O.BFLOAT16: 2, O.FLOAT16: 2, O.F8E4M3: 1, O.F8E5M2: 1, O.INT8: 1}
N = 3 * 8192 + 4099  # past three of the largest chunk (8192 Int4 elements), odd
PADS = [(0, 2), (2, 0), (1, 4), (3, 6), (8, 12), (5, 1)]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    M.init(0)


def run(call, src, out_bytes, pads):
    """The bytes `call(out pointer, in pointer)` writes, with a guard of 64 bytes after them."""
    st, sp = to_dev(src, pad=pads[0])
    ot, op = empty_dev(out_bytes + 64, pad=pads[1])
    call(op, sp)
    got = to_host(ot, np.uint8)
    assert (got[:pads[1]] == 0xA5).all() and (got[pads[1] + out_bytes:] == 0xA5).all(), "wrote outside the output"
    return got[pads[1]:pads[1] + out_bytes]


def same(got, want, what):
    w = np.ascontiguousarray(want).view(np.uint8).reshape(-1)
    bad = np.flatnonzero(got != w)
    assert bad.size == 0, f"{what}: {bad.size} bytes differ, first at {bad[0]}"


@pytest.mark.parametrize("pads", PADS)
@pytest.mark.parametrize("out_dt", [O.BFLOAT16, O.FLOAT32])
def test_fp8_and_int4_dequant(out_dt, pads):
    rng = np.random.default_rng(out_dt + pads[0])
    codes = rng.integers(0, 256, N, dtype=np.uint8)
    got = run(lambda o, i: M.dequant_fp8(o, out_dt, i, O.F8E4M3, N, 0.0125, stream()), codes, N * SIZE[out_dt], pads)
    same(got, O.dequant_fp8(codes, O.F8E4M3, float(np.float32(0.0125)), out_dt), f"fp8 {pads}")
    packed = rng.integers(0, 256, (N + 1) // 2, dtype=np.uint8)
    scales = O.f32_to_f16(rng.uniform(0.005, 0.02, N // 128 + 1).astype(np.float32))
    sct, scp = to_dev(scales, pad=2)
    got = run(lambda o, i: M.dequant_int4(o, out_dt, i, N, scp, O.FLOAT16, 128, stream()), packed, N * SIZE[out_dt], pads)
    same(got, O.dequant_int4(packed, N, scales, O.FLOAT16, 128, out_dt), f"int4 {pads}")


def source(dt, rng):
    if dt in (O.INT8, O.F8E4M3, O.F8E5M2):
        return rng.integers(0, 256, N, dtype=np.uint8)
    v = rng.normal(0, 40, N)
    return v if dt == O.FLOAT64 else O.encode(v.astype(np.float32), dt)


@pytest.mark.parametrize("pads", PADS)
@pytest.mark.parametrize("in_dt, out_dt", [
    (O.FLOAT32, O.BFLOAT16), (O.BFLOAT16, O.FLOAT32), (O.FLOAT16, O.BFLOAT16), (O.FLOAT64, O.FLOAT32),
    (O.FLOAT64, O.FLOAT16), (O.INT8, O.FLOAT32), (O.FLOAT32, O.FLOAT32), (O.FLOAT32, O.FLOAT64),
    (O.BFLOAT16, O.FLOAT64), (O.FLOAT32, O.F8E4M3), (O.BFLOAT16, O.F8E4M3), (O.FLOAT64, O.INT8),
    (O.INT8, O.INT8), (O.F8E5M2, O.INT8), (O.F8E4M3, O.F8E5M2)])
def test_casts(in_dt, out_dt, pads):
    a = source(in_dt, np.random.default_rng(in_dt * 16 + out_dt + pads[0]))
    if in_dt == O.INT8:
        a = a.view(np.int8)
    got = run(lambda o, i: M.convert(o, out_dt, i, in_dt, N, stream()), a, N * SIZE[out_dt], pads)
    want = {O.FLOAT64: O.bytes_to_f64, O.FLOAT32: O.bytes_to_f32, O.BFLOAT16: O.bytes_to_bf16, O.FLOAT16: O.bytes_to_f16,
            O.INT8: O.bytes_to_i8}.get(out_dt)
    want = want(in_dt, a) if want else O.f32_to_fp8(O.bytes_to_f32(in_dt, a), out_dt)
    same(got, want, f"{in_dt}->{out_dt} {pads}")


@pytest.mark.parametrize("pads", PADS)
@pytest.mark.parametrize("in_dt", [O.FLOAT32, O.FLOAT16, O.INT8, O.FLOAT64, O.F8E4M3])
def test_int4_encode(in_dt, pads):
    a = source(in_dt, np.random.default_rng(in_dt + pads[1]))
    if in_dt == O.INT8:
        a = a.view(np.int8)
    got = run(lambda o, i: M.convert(o, O.INT4, i, in_dt, N, stream()), a, (N + 1) // 2, pads)
    same(got, O.bytes_to_i4(in_dt, a, N), f"{in_dt}->i4 {pads}")


@pytest.mark.parametrize("pads", PADS)
@pytest.mark.parametrize("dt", [O.FLOAT32, O.BFLOAT16, O.FLOAT16])
def test_axpy_broadcast_linspace(dt, pads):
    rng = np.random.default_rng(dt + pads[0])
    x, y = (O.encode(rng.normal(0, 3, N).astype(np.float32), dt) for _ in range(2))
    xt, xp = to_dev(x, pad=pads[0])

    def axpy(o, i):
        M.axpy(i, xp, N, -1.3, dt, stream())
        M.stream_sync(stream())

    yt, yp = to_dev(y, pad=pads[1])
    axpy(0, yp)
    same(to_host(yt, np.uint8)[pads[1]:], O.axpy_storage(y, x, -1.3, dt), f"axpy {dt} {pads}")
    got = run(lambda o, i: M.scalar_broadcast(o, dt, i, dt, N, 0.37, "mul", stream()), x, N * SIZE[dt], pads)
    same(got, O.encode(O.scalar_broadcast(O.decode(x, dt), 0.37, "mul"), dt), f"broadcast {dt} {pads}")
    got = run(lambda o, i: M.linspace(o, dt, N, -3.5, 11.0, True, stream()), x, N * SIZE[dt], pads)
    same(got, O.encode(O.linspace(-3.5, 11.0, N, True), dt), f"linspace {dt} {pads}")


@pytest.mark.parametrize("pads", PADS[:4])
@pytest.mark.parametrize("n", [1, 31, 4095, 4096, 4097, 3 * 4096 + 33])
@pytest.mark.parametrize("out_dt", [O.F8E4M3, O.F8E5M2, O.INT8, O.INT4])
def test_int4_sources_by_table(out_dt, n, pads):
    # whole 16-nibble pieces and the element tail; every byte value
    packed = np.resize(np.random.default_rng(n).permutation(256).astype(np.uint8), (n + 1) // 2)
    got = run(lambda o, i: M.convert(o, out_dt, i, O.INT4, n, stream()), packed,
              (n + 1) // 2 if out_dt == O.INT4 else n, pads)
    if out_dt == O.INT4:
        want = O.bytes_to_i4(O.INT4, packed, n)
    elif out_dt == O.INT8:
        want = O.bytes_to_i8(O.INT4, packed)[:n]
    else:
        want = O.f32_to_fp8(O.bytes_to_f32(O.INT4, packed), out_dt)[:n]
    same(got, want, f"i4->{out_dt} n={n} {pads}")


@pytest.mark.parametrize("in_dt", [O.F8E4M3, O.F8E5M2])
@pytest.mark.parametrize("out_dt", [O.F8E4M3, O.F8E5M2, O.INT8, O.INT4])
def test_fp8_sources_every_code(in_dt, out_dt):
    # every code, NaN and infinities among them, through whole pieces and the tail
    n = 2 * 4096 + 77
    a = np.resize(np.arange(256, dtype=np.uint8), n)
    got = run(lambda o, i: M.convert(o, out_dt, i, in_dt, n, stream()), a, (n + 1) // 2 if out_dt == O.INT4 else n, (0, 0))
    want = (O.bytes_to_i4(in_dt, a, n) if out_dt == O.INT4 else O.bytes_to_i8(in_dt, a) if out_dt == O.INT8
            else O.f32_to_fp8(O.bytes_to_f32(in_dt, a), out_dt))
    same(got, want, f"{in_dt}->{out_dt}")


@pytest.mark.parametrize("pads", [(0, 0), (1, 1)])
@pytest.mark.parametrize("out_dt", [O.F8E4M3, O.INT8, O.INT4])
@pytest.mark.parametrize("in_dt", [O.FLOAT64, O.FLOAT32, O.BFLOAT16, O.INT8, O.F8E5M2, O.INT4])
def test_encode_wave_split(in_dt, out_dt, pads):
    # 64 pieces per wave, from 2^17 pieces on whole chunks of 256 first, then fewer elements than a piece
    piece = 16 // SIZE.get(in_dt, 1)
    counts = [pieces * piece + d for pieces in (0, 1, 63, 64, 65, 256, 257) for d in (-1, 0, 1, piece // 2)]
    counts += [(1 << 17) * piece - 1, (1 << 17) * piece, ((1 << 17) + 256 + 65) * piece + 1]
    for n in sorted({n for n in counts if n > 0}):
        rng = np.random.default_rng(n)
        if in_dt == O.INT4:
            a = rng.integers(0, 256, (n + 1) // 2, dtype=np.uint8)
        elif in_dt == O.INT8:
            a = rng.integers(-128, 128, n).astype(np.int8)
        else:
            a = rng.integers(0, 256, n, dtype=np.uint8) if in_dt == O.F8E5M2 else rng.normal(0, 40, n)
            a = O.encode(a.astype(np.float32), in_dt) if in_dt in (O.FLOAT32, O.BFLOAT16) else a
        got = run(lambda o, i: M.convert(o, out_dt, i, in_dt, n, stream()), a, (n + 1) // 2 if out_dt == O.INT4 else n, pads)
        want = (O.bytes_to_i4(in_dt, a, n) if out_dt == O.INT4 else O.bytes_to_i8(in_dt, a)[:n] if out_dt == O.INT8
                else O.f32_to_fp8(O.bytes_to_f32(in_dt, a), out_dt)[:n])
        same(got, want, f"{in_dt}->{out_dt} n={n} {pads}")
