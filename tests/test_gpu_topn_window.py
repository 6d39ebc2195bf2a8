"""TopN selections that start from the boundary of the one before (one pass over the keys and a rank among the few
collected) against the ordering computed in numpy: larger |c|^2 first, then the reference's canonical order, a NaN never.
Each sum is cut several times in a row, so that every cut but the first has a boundary to start from: by a few terms and
by most of them, through distinct coefficients, runs of equal ones around the ranking's limits (1024 and 2048), NaNs and
infinities.  Sums below and above the size from which the window is narrowed by a launch of its own."""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_transfer import canonical, distinct, upload

pytestmark = pytest.mark.gpu


def kept(num_qubits, x, z, c, bits, n):
    x, z, c = canonical(num_qubits, x, z, c, bits)
    with np.errstate(over="ignore", invalid="ignore"):
        u = c.astype(np.float64) ** 2
    finite = ~np.isnan(u)
    if len(c) <= n:
        return x, z, c
    order = np.argsort(-np.where(finite, u, -1.0), kind="stable")  # stable: canonical among equals
    stay = np.zeros(len(c), bool)
    stay[order[:n]] = True
    stay &= finite
    return x[stay], z[stay], c[stay]


def coefficients(rng, n, values, dtype):
    c = rng.standard_normal(n)
    if values == "digits":  # runs of about n / 400 equal magnitudes of either sign
        c = np.round(c, 2) + 0.001
        c[rng.random(n) < 0.5] *= -1
    elif values == "runs":  # runs of 1024, 1025, 2048, 2049 and 5000 equal ones among distinct ones
        at = 0
        for k, run in enumerate((1024, 1025, 2048, 2049, 5000)):
            c[at:at + run] = 0.5 + 0.1 * k
            at += run
    elif values == "equal":
        c[:] = 0.25
    elif values == "special":
        c[rng.random(n) < 0.05] = np.nan
        c[rng.random(n) < 0.05] = np.inf
        c[rng.random(n) < 0.05] = -np.inf
    return c.astype(dtype)


@pytest.mark.parametrize("num_qubits,dtype", [(50, np.float64), (127, np.float64), (64, np.float32), (100, np.float32)])
@pytest.mark.parametrize("values", ["distinct", "digits", "runs", "equal", "special"])
@pytest.mark.parametrize("n", [3_000, 40_000])
def test_cuts_in_a_row(num_qubits, dtype, values, n):
    if values == "runs" and n < 12_000:
        pytest.skip("the runs do not fit")
    rng = np.random.default_rng([num_qubits, n])
    x, z, _ = distinct(rng, n, num_qubits, dtype)
    c = coefficients(rng, n, values, dtype)
    g = upload(num_qubits, x, z, c)
    bits = g.bucket_bits()[0]
    try:
        for cut in (n - 3, n - 4, n - n // 50, n - n // 20, n - n // 6, n // 2, n // 2 - 1, n // 2 - n // 40, n // 9, 2, 1):
            g.truncate_topn(cut)
            x, z, c = kept(num_qubits, x, z, c, bits, cut)
            h = g.to_host()
            assert len(h) == len(c), cut
            assert np.array_equal(h._x, x) and np.array_equal(h._z, z) and np.array_equal(h._c, c, equal_nan=True), cut
        assert all(v == 0 for k, v in g.check_layout().items() if k != "unscanned")
    finally:
        g.free()


@pytest.mark.parametrize("num_qubits,dtype,values", [(60, np.float64, "distinct"), (127, np.float32, "digits"),
                                                     (127, np.float64, "runs")])
@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, 700_001])
def test_cuts_of_larger_sums(num_qubits, dtype, values, n):
    rng = np.random.default_rng([num_qubits, n])
    x, z, _ = distinct(rng, n, num_qubits, dtype)
    c = coefficients(rng, n, values, dtype)
    g = upload(num_qubits, x, z, c)
    bits = g.bucket_bits()[0]
    try:
        for cut in (n - 100, n - n // 100, n - n // 25, n - n // 24, n // 3):
            g.truncate_topn(cut)
            x, z, c = kept(num_qubits, x, z, c, bits, cut)
            h = g.to_host()
            assert np.array_equal(h._x, x) and np.array_equal(h._z, z) and np.array_equal(h._c, c), cut
    finally:
        g.free()
