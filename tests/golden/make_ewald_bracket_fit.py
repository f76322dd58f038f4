"""Generator of the Ewald force bracket of the pair kernels' force-only path.

The direct Coulomb force factor of a pair is
  qq B(beta r) / r^3,   B(x) = erfc(x) + 2/sqrt(pi) x exp(-x^2),
with B falling from 1 to 7.7e-4 on 0 <= x <= sqrt(8.5).  B is evaluated as the
square of a polynomial of degree 14 in s = 2 x / sqrt(8.5) - 1: sqrt(B) falls to
0.028 only, so the polynomial's FP32 rounding (half an ulp of the largest partial
sum, 3e-8) is 1e-6 of it at the far end where it is 4e-5 of B itself, and no two
nearly equal numbers are subtracted.  The fit's relative error is weighted by
min(1, 10^(0.8 (1 - x))): a pair's force falls as B / x^2, by a factor of 1e4
between x = 1 and the far end, so an error there weighs less in a sum.  The
coefficients minimise the largest weighted error by Lawson's algorithm
(iteratively reweighted least squares) over 3000 Chebyshev-spaced samples, in
FP64 against scipy's erfc.

Run:  python tests/golden/make_ewald_bracket_fit.py
prints the coefficients (highest power first, the order of the kernel's Horner
evaluation) and the largest weighted error of the fit in FP64.
"""
from __future__ import annotations

import numpy as np
from scipy.special import erfc

Z_MAX = 8.5
X_MAX = float(np.sqrt(Z_MAX))
DEGREE = 14
SLOPE = 0.8


def bracket(x):
    x = np.asarray(x, np.float64)
    return erfc(x) + 2.0 / np.sqrt(np.pi) * x * np.exp(-x * x)


def weight(x):
    return np.minimum(1.0, 10.0 ** (SLOPE * (1.0 - np.asarray(x, np.float64))))


def samples(n=3000):
    k = np.arange(n)
    return np.cos(np.pi * (k + 0.5) / n)  # s


def fit(iterations=300):
    """Coefficients c[p] of s^p (lowest first)."""
    s = samples()
    x = 0.5 * X_MAX * (s + 1.0)
    y = np.sqrt(bracket(x))
    W = weight(x) / y
    V = np.polynomial.chebyshev.chebvander(s, DEGREE)
    lawson = np.full(len(s), 1.0 / len(s))
    c = None
    for _ in range(iterations):
        sw = np.sqrt(lawson) * W
        c, *_ = np.linalg.lstsq(V * sw[:, None], y * sw, rcond=None)
        lawson = lawson * (np.abs((V @ c - y) * W) + 1e-300)
        lawson /= lawson.sum()
    return np.polynomial.chebyshev.cheb2poly(c)


def max_weighted_error(c_low_first, n=20000):
    """Largest weighted relative error of the squared polynomial in FP64."""
    s = samples(n)
    x = 0.5 * X_MAX * (s + 1.0)
    p = np.polynomial.polynomial.polyval(s, np.asarray(c_low_first, np.float64))
    return float(np.max(np.abs(p * p / bracket(x) - 1.0) * weight(x)))


def evaluate32(c_high_first, s):
    """FP32 evaluation as in the kernel: Horner by fused multiply-adds, squared."""
    r32 = lambda v: np.asarray(v).astype(np.float32).astype(np.float64)  # noqa: E731
    p = np.full_like(s, float(np.float32(c_high_first[0])))
    for v in c_high_first[1:]:
        p = r32(p * s + float(np.float32(v)))
    return r32(p * p)


if __name__ == "__main__":
    c = fit()
    print("coefficients, highest power of s first (Horner order of the kernel):")
    for v in c[::-1]:
        print(f"    {float(np.float32(v)):.9e}")
    print(f"max weighted error on [0, {X_MAX:.4f}]: {max_weighted_error(c):.3e}, "
          f"of the FP32 coefficients {max_weighted_error(c.astype(np.float32)):.3e}")
