"""The Ewald force polynomial of the learned form's pair field
(sponge_amd/csrc/common.h, kEwaldForce) against scipy, its FP32 Horner
evaluation, and its generator (tests/golden/make_ewald_force_fit.py)
reproducing a fit of the same accuracy."""
import os
import re
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests", "golden"))

import make_ewald_force_fit as G  # noqa: E402


def committed_coefficients():
    """kEwaldForce in Horner order (highest power of s first)."""
    src = open(os.path.join(ROOT, "sponge_amd", "csrc", "common.h")).read()
    body = src[src.index("constexpr float kEwaldForce["):]
    body = body[:body.index("};")]
    vals = re.findall(r"([-+]?\d\.\d+e[-+]\d+)f", body)
    assert len(vals) == G.DEGREE + 1, vals
    zmax = re.search(r"constexpr float kEwaldZMax = ([0-9.]+)f;", src)
    assert zmax and float(zmax.group(1)) == G.Z_MAX
    return [float(v) for v in vals]


def test_committed_constants_fp64():
    err = G.max_weighted_error(committed_coefficients()[::-1])
    print(f"FP64 max weighted error {err:.3e}")
    assert err < 9e-9


def test_committed_constants_fp32_horner():
    c = np.asarray(committed_coefficients(), np.float32).astype(np.float64)
    s = G.samples(20000).astype(np.float32).astype(np.float64)
    p = np.full_like(s, c[0])
    for v in c[1:]:  # fused multiply-adds: one FP32 rounding per step
        p = (p * s + v).astype(np.float32).astype(np.float64)
    err = np.abs(p - G.H(0.5 * G.Z_MAX * (s + 1.0)))
    print(f"FP32 Horner max absolute error {err.max():.3e}")
    # H falls from 0.75 to 0.04: half an ulp of the value at z = 0 bounds the
    # rounding; the fit's own error below z = 2 is weighted (see the generator)
    assert (err * G.weight(0.5 * G.Z_MAX * (s + 1.0))).max() < 1.2e-7
    # the outer half, where the force factor is a difference of nearly equal
    # terms (values below 0.11, ulp 7.5e-9)
    assert err[s > 0].max() < 2.5e-8


def test_generator_reproduces_the_fit():
    c = G.fit()
    assert G.max_weighted_error(c) < 1.5e-8
    committed = np.asarray(committed_coefficients()[::-1])
    assert np.max(np.abs(c - committed)) < 1e-7
