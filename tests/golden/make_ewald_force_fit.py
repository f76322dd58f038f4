"""Generator of the Ewald force polynomial of the learned form's pair field.

The reciprocal part of an Ewald pair's force,
  H(z) = (erf(x) - 2/sqrt(pi) x exp(-x^2)) / x^3,  z = x^2,
is entire in z; the force factor of a pair is qq beta^3 H(beta^2 r^2), and the
direct part is the difference to qq / r^3, so neither needs an exponential.  H
is fitted on 0 <= z <= 8.5 by a polynomial of degree 12 in s = 2 z / 8.5 - 1 (in
s, not z: the coefficients fall geometrically, so FP32 Horner evaluation stays
at the rounding of the result).  The error is weighted by what it does to the
direct force: beyond z = 2 by its absolute size, below by its size against the
1/x^3 that H is subtracted from (weight min(1, x^3 / 3)); relative to H itself
it is 6e-7 at x = 0.275 and 1e-6 at half of that.  The coefficients minimise the
largest weighted error by Lawson's algorithm (iteratively reweighted least
squares) over 4000 Chebyshev-spaced samples, in FP64 against scipy's confluent
hypergeometric function: H(z) = 4 / (3 sqrt(pi)) 1F1(3/2; 5/2; -z).

Run:  python tests/golden/make_ewald_force_fit.py
prints the coefficients (highest power first, the order of the kernel's Horner
evaluation) and the largest weighted error of the fit in FP64.
"""
from __future__ import annotations

import math

import numpy as np
from scipy.special import hyp1f1

Z_MAX = 8.5
DEGREE = 12


def H(z):
    return 4.0 / (3.0 * math.sqrt(math.pi)) * hyp1f1(1.5, 2.5, -np.asarray(z, np.float64))


def samples(n=4000):
    k = np.arange(n)
    return -np.cos(np.pi * (k + 0.5) / n)  # s


def weight(z):
    return np.minimum(1.0, np.asarray(z, np.float64) ** 1.5 / 3.0)


def fit(iterations=300):
    """Coefficients c[p] of s^p (lowest first)."""
    s = samples()
    z = 0.5 * Z_MAX * (s + 1.0)
    W = weight(z)
    A = np.polynomial.chebyshev.chebvander(s, DEGREE) * W[:, None]
    b = H(z) * W
    w = np.full(len(s), 1.0 / len(s))
    c = None
    for _ in range(iterations):
        sw = np.sqrt(w)
        c, *_ = np.linalg.lstsq(A * sw[:, None], b * sw, rcond=None)
        w = w * np.abs(A @ c - b)
        w /= w.sum()
    return np.polynomial.chebyshev.cheb2poly(c)


def max_weighted_error(c_low_first):
    s = samples(20000)
    z = 0.5 * Z_MAX * (s + 1.0)
    p = np.polynomial.polynomial.polyval(s, np.asarray(c_low_first, np.float64))
    return float(np.max(np.abs(p - H(z)) * weight(z)))


def horner32(c_high_first, s):
    """FP32 Horner evaluation by fused multiply-adds (one rounding per step)."""
    p = np.full_like(s, c_high_first[0])
    for v in c_high_first[1:]:
        p = (p * s + v).astype(np.float32).astype(np.float64)
    return p


def round_coefficients(c_low_first, sweeps=4):
    """FP32 coefficients (highest power first): each in turn moved by an ulp
    while that lowers the largest weighted error of the FP32 evaluation (plain
    rounding of all 13 alone costs 1.4e-8 at s = 1)."""
    s = samples(2000).astype(np.float32).astype(np.float64)
    z = 0.5 * Z_MAX * (s + 1.0)
    ref, W = H(z), weight(z)
    c = np.asarray(c_low_first, np.float64)[::-1].astype(np.float32)

    def err(v):
        return float(np.max(np.abs(horner32(v.astype(np.float64), s) - ref) * W))

    best = err(c)
    for _ in range(sweeps):
        for k in range(len(c)):
            for up in (np.float32(np.inf), np.float32(-np.inf)):
                t = c.copy()
                t[k] = np.nextafter(c[k], up)
                if err(t) < best:
                    c, best = t, err(t)
    return c


if __name__ == "__main__":
    c = round_coefficients(fit())[::-1]
    print("coefficients, highest power of s first (Horner order of the kernel):")
    for v in c[::-1]:
        print(f"    {v:.9e}")
    print(f"max weighted error on [0, {Z_MAX}]: {max_weighted_error(c):.3e}")
