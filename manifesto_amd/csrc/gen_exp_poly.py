"""Derives the constants of the f32 exponential kernels in devmath.hpp.

e^x = 2^k * e^r with k = rint(x / ln2) and r = x - k*ln2 (Cody & Waite range
reduction, ln2 split into a 16-bit head, so k*head is exact for |k| < 256, and
an f32 tail).  e^r on |r| <= ln2/2 (plus a margin for the f32 rounding of
x/ln2) is a degree-6 polynomial with the constant term pinned to 1, fitted by
weighted least squares on Chebyshev nodes for relative error and rounded to
f32.

2^f on |f| <= 1/2 (the fraction left when the argument is already in log2
units and reduced in f64) is fitted the same way, once with f32 coefficients
(degree 6, within 0.94 f32 ulp; gelu now uses the hardware v_exp_f32
instead, which measured faster and equally accurate) and once with f64
coefficients (degree 8, fitted in 50-digit arithmetic with mpmath; sigmoid).

Two more f64 fits, by the same weighted least squares in 50 digits, serve tanh
and log: 2^f - 1 = f q(f) of degree 9, relative to 2^f - 1 for f > 0 and to
2^(1 + f) - 1 for f < 0 (fit_expm1_f64), and (2 atanh(s) - 2 s) / s^3 as a
polynomial of degree 4 in s^2 for |s| <= (sqrt(2) - 1) / (sqrt(2) + 1)
(fit_log_f64).

Run: python3 gen_exp_poly.py
"""
import math

import numpy as np

F32 = np.float32


def f32_hex(v):
    return "0x%08xu" % int(np.array([v], dtype=np.float32).view(np.uint32)[0])


def split_ln2():
    ln2 = math.log(2.0)
    head = math.floor(ln2 * 2 ** 16) / 2 ** 16  # 16 significant bits
    tail = float(F32(ln2 - head))
    return F32(head), F32(tail)


def fit(degree=6, half_width=0.3466 + 2e-5, nodes=4000):
    k = np.arange(nodes)
    r = half_width * np.cos(np.pi * (k + 0.5) / nodes)
    target = np.expm1(r)  # fit e^r - 1 = r * q(r), q of degree-1
    basis = np.stack([r ** (j + 1) for j in range(degree)], axis=1)
    w = 1.0 / np.exp(r)
    coef, *_ = np.linalg.lstsq(basis * w[:, None], target * w, rcond=None)
    return [F32(c) for c in coef]


def fit_exp2(degree=6, half_width=0.5, nodes=4000):
    k = np.arange(nodes)
    f = half_width * np.cos(np.pi * (k + 0.5) / nodes)
    target = np.expm1(f * math.log(2.0))  # 2^f - 1 = f * q(f)
    basis = np.stack([f ** (j + 1) for j in range(degree)], axis=1)
    w = 1.0 / np.exp2(f)
    coef, *_ = np.linalg.lstsq(basis * w[:, None], target * w, rcond=None)
    return [F32(c) for c in coef]


def fit_exp2_f64(degree=8, half_width=0.5, nodes=600):
    """Weighted least squares for 2^f - 1 = f q(f) in 50-digit arithmetic;
    returns the coefficients rounded to f64 and the max relative error of
    the f64 Horner evaluation on a grid."""
    import mpmath as mp
    mp.mp.dps = 50
    xs = [half_width * mp.cos(mp.pi * (k + mp.mpf(0.5)) / nodes) for k in range(nodes)]
    A = mp.matrix(nodes, degree)
    b = mp.matrix(nodes, 1)
    for i, x in enumerate(xs):
        w = 1 / mp.power(2, x)
        for j in range(degree):
            A[i, j] = w * x ** (j + 1)
        b[i] = w * (mp.power(2, x) - 1)
    Q, R = mp.qr(A)
    c = mp.lu_solve(R[:degree, :degree], (Q.T * b)[:degree, 0])
    coef = [float(c[j]) for j in range(degree)]
    worst = 0
    for i in range(4001):
        f = -half_width + 2 * half_width * i / 4000
        acc = coef[-1]
        for cj in reversed(coef[:-1]):
            acc = acc * f + cj
        acc = acc * f + 1.0
        worst = max(worst, abs((mp.mpf(acc) - mp.power(2, mp.mpf(f))) / mp.power(2, mp.mpf(f))))
    return coef, float(mp.log(worst, 2))


def lsq_f64(xs, basis, target, weight):
    """Weighted least squares in mpmath arithmetic, coefficients rounded to f64."""
    import mpmath as mp
    n, d = len(xs), len(basis(xs[0]))
    A, b = mp.matrix(n, d), mp.matrix(n, 1)
    for i, x in enumerate(xs):
        w = weight(x)
        for j, v in enumerate(basis(x)):
            A[i, j] = w * v
        b[i] = w * target(x)
    Q, R = mp.qr(A)
    c = mp.lu_solve(R[:d, :d], (Q.T * b)[:d, 0])
    return [float(c[j]) for j in range(d)]


def chebyshev(a, b, n):
    import mpmath as mp
    return [(a + b) / 2 + (b - a) / 2 * mp.cos(mp.pi * (k + mp.mpf(0.5)) / n) for k in range(n)]


def fit_expm1_f64(degree=9):
    """tanh: coefficients of f q(f) and the largest weighted error."""
    import mpmath as mp
    mp.mp.dps = 50
    two = mp.mpf(2)

    def weight(f):
        return 1 / (two ** f - 1) if f > 0 else 2 / (two ** (1 + f) - 1)

    xs = chebyshev(mp.mpf(-0.5), mp.mpf(0.5), 400)
    c = lsq_f64(xs, lambda f: [f ** (j + 1) for j in range(degree)], lambda f: two ** f - 1, weight)
    worst = 0
    for i in list(range(-2000, 0)) + list(range(1, 2001)):
        f = mp.mpf(i) / 4000
        acc = mp.mpf(0)
        for cj in reversed(c):
            acc = (acc + cj) * f
        worst = max(worst, abs(acc - (two ** f - 1)) * weight(f))
    return c, float(mp.log(worst, 2))


def fit_log_f64(terms=5):
    """log: coefficients in s^2 and the largest error relative to 2 atanh(s)."""
    import mpmath as mp
    mp.mp.dps = 50
    top = ((mp.sqrt(2) - 1) / (mp.sqrt(2) + 1)) ** 2
    c = lsq_f64(chebyshev(mp.mpf(0), top, 200), lambda y: [y ** j for j in range(terms)],
                lambda y: (2 * mp.atanh(mp.sqrt(y)) - 2 * mp.sqrt(y)) / mp.sqrt(y) ** 3, lambda y: y)
    worst = 0
    for i in range(1, 2001):
        y = top * i / 2000
        s = mp.sqrt(y)
        acc = mp.mpf(0)
        for cj in reversed(c):
            acc = acc * y + cj
        worst = max(worst, abs((2 * s + s * y * acc) / (2 * mp.atanh(s)) - 1))
    return c, float(mp.log(worst, 2))


def horner_f32(coef, r):
    """Evaluates 1 + r*(c1 + r*(c2 + ...)) with f32 fma rounding."""
    r64 = r.astype(np.float64)
    acc = np.full_like(r, coef[-1], dtype=np.float32)
    for c in reversed(coef[:-1]):
        acc = (acc.astype(np.float64) * r64 + float(c)).astype(np.float32)
    return (acc.astype(np.float64) * r64 + 1.0).astype(np.float32)


def main():
    head, tail = split_ln2()
    coef = fit()
    r = np.linspace(-0.3467, 0.3467, 2_000_001).astype(np.float32)
    approx = horner_f32(coef, r).astype(np.float64)
    exact = np.exp(r.astype(np.float64))
    ulp = np.spacing(exact.astype(np.float32)).astype(np.float64)
    err = np.abs(approx - exact) / ulp
    print("ln2 head", f32_hex(head), float(head))
    print("ln2 tail", f32_hex(tail), float(tail))
    for j, c in enumerate(coef, start=1):
        print(f"c{j}", f32_hex(c), repr(float(c)))
    print("max error of e^r in f32 ulps (incl. Horner rounding):", err.max())
    coef2 = fit_exp2()
    f = np.linspace(-0.5, 0.5, 2_000_001).astype(np.float32)
    approx = horner_f32(coef2, f).astype(np.float64)
    exact = np.exp2(f.astype(np.float64))
    err = np.abs(approx - exact) / np.spacing(exact.astype(np.float32)).astype(np.float64)
    for j, c in enumerate(coef2, start=1):
        print(f"2^f c{j}", f32_hex(c), repr(float(c)))
    print("max error of 2^f in f32 ulps (incl. Horner rounding):", err.max())
    try:
        coef64, log2err = fit_exp2_f64()
    except ImportError:
        print("mpmath is not installed: f64 coefficients skipped")
        return
    for j, c in enumerate(coef64, start=1):
        print(f"2^f f64 c{j}", float.hex(c))
    print("log2 of the max relative error of 2^f in f64:", log2err)
    for name, fit_f64 in (("2^f - 1 (tanh)", fit_expm1_f64), ("log", fit_log_f64)):
        coefs, log2err = fit_f64()
        for j, c in enumerate(coefs):
            print(f"{name} coefficient {j}", float.hex(c))
        print(f"log2 of the max weighted error of {name}:", log2err)


if __name__ == "__main__":
    main()
