"""The Ewald force bracket of the pair kernels' force-only path
(sponge_amd/csrc/common.h, kBracket) against scipy, its FP32 evaluation, and its
generator (tests/golden/make_ewald_bracket_fit.py) reproducing the fit.

FP32 bounds: the polynomial's evaluation errs by a few half ulps of numbers below
one (9e-8), twice that over its value relative to its square, beside the fit's
own weighted error: 1e-6 where x < 1 (value above 0.87), 1.2e-5 at the far end
(value 0.028, weight 1/34)."""
import os
import re
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests", "golden"))

import make_ewald_bracket_fit as G  # noqa: E402


def committed_coefficients():
    """kBracket in Horner order (highest power of s first)."""
    src = open(os.path.join(ROOT, "sponge_amd", "csrc", "common.h")).read()
    body = src[src.index("constexpr float kBracket["):]
    body = body[:body.index("};")]
    vals = re.findall(r"([-+]?\d\.\d+e[-+]\d+)f", body)
    assert len(vals) == G.DEGREE + 1, vals
    xmax = re.search(r"constexpr float kBracketXMax = ([0-9.]+)f;", src)
    assert xmax and np.float32(float(xmax.group(1))) == np.float32(G.X_MAX)
    return [float(v) for v in vals]


def test_committed_constants_fp64():
    err = G.max_weighted_error(committed_coefficients()[::-1])
    print(f"FP64 max weighted relative error {err:.3e}")
    assert err < 2e-7


def test_committed_constants_fp32():
    s = np.linspace(-1.0, 1.0, 40001).astype(np.float32).astype(np.float64)
    x = 0.5 * G.X_MAX * (s + 1.0)
    err = np.abs(G.evaluate32(committed_coefficients(), s) / G.bracket(x) - 1.0)
    print(f"FP32 max relative error {err[x < 1].max():.3e} below x = 1, {err.max():.3e}")
    assert err[x < 1].max() < 1e-6
    assert err.max() < 1.2e-5


def test_generator_reproduces_the_fit():
    c = G.fit()
    assert G.max_weighted_error(c) < 1e-7
    assert np.max(np.abs(c - np.asarray(committed_coefficients()[::-1]))) < 1e-7
