"""Learned selections in a row on one sum whose boundary passes through a score of zero: a window around it spans most of
the score keys' range (their order-mapped bits run through both signs' exponents).  With a network of zero weights the
score is ln|c| alone, so the boundary is chosen through the coefficients: below, at and above zero, by one term and by
many, with runs of equal scores, below and above the size from which a window is narrowed by a launch of its own.  The
kept terms are those of the order computed in numpy."""

from __future__ import annotations

import numpy as np
import pytest

from paulistrings_amd import Circuit, truncation
from paulistrings_amd import learned as PL
from test_gpu_transfer import canonical, distinct, upload

pytestmark = pytest.mark.gpu


def score_is_ln_c():
    m = PL.Model(PL.lattice_groups(8, 8), depth_scale=40.0, seed=1)
    m.set_params(np.zeros(PL.Model.param_count(), np.float32))
    return m


@pytest.mark.parametrize("n", [6_000, 600_000])
@pytest.mark.parametrize("runs", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_cuts_across_score_zero(n, runs, dtype):
    rng = np.random.default_rng([n, runs])
    x, z, _ = distinct(rng, n, 64, dtype)
    c = np.exp(np.linspace(-2.0, 2.0, n))  # scores 4 / n apart, far more than a float's rounding
    if runs:  # a hundredth of the terms share each score: exactly 1, and one on either side of it
        for k, at in enumerate((0.3, 0.5, 0.7)):
            c[int(at * n):int(at * n) + n // 100] = (0.45, 1.0, 2.2)[k]
    c = rng.permutation(c * rng.choice([-1.0, 1.0], n)).astype(dtype)
    m = score_is_ln_c()
    g = upload(64, x, z, c)
    try:
        bits = g.bucket_bits()[0]
        cx, cz, cc = canonical(64, x, z, c, bits)
        order = np.argsort(-np.log(np.abs(cc.astype(np.float64))), kind="stable")  # stable: canonical among equals
        # boundaries at about these scores, each cut again by one term and by 1/300 of what is left
        for score in (-1.5, -0.8, -0.71, -0.3, -0.1, -0.02, 0.0, 0.01, 0.1, 0.5, 0.69, 0.72, 1.39, 1.41, 1.9):
            at = int(n * (2.0 - score) / 4.0)
            for keep in (at, at - 1, at - 1 - at // 300):
                PL.truncate_learned(g, m, keep, 3.0)
                stay = np.sort(order[:keep])
                h = g.to_host()
                assert np.array_equal(h._x, cx[stay]) and np.array_equal(h._z, cz[stay]), (score, keep)
                assert np.array_equal(h._c, cc[stay]), (score, keep)
    finally:
        g.free()
        m.free()


def test_propagation_with_its_boundary_near_score_zero(monkeypatch):
    rng = np.random.default_rng(8)
    n, keep = 5_000, 2_500
    x, z, _ = distinct(rng, n, 36, np.float64)
    c = np.exp(rng.uniform(-0.5, 0.5, n))
    circ = Circuit(36)
    for q in range(30):
        circ.rx(0.05 + 0.001 * q, q)
        circ.rzz(0.04, q, q + 1)
    m = score_is_ln_c()
    out = []
    for window in ("1", "0"):
        monkeypatch.setenv("PP_TOPN_WINDOW", window)
        g = upload(36, x, z, c)
        PL.propagate_learned(g, circ, m, keep, truncation.coeff(1e-8), "heisenberg")
        out.append(g.to_host())
        g.free()
    m.free()
    a, b = out
    assert len(a) == keep
    assert np.array_equal(a._x, b._x) and np.array_equal(a._z, b._z) and np.array_equal(a._c, b._c)
