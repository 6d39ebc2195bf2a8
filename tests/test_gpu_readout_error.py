"""A read-out's error against the exact sum (math.fsum): the sum rounded once, whatever its order and cancellation.  A sum
of n numbers that carries the error of each of its additions is off by at most u |S| + (n u)^2 sum |c| with u = 2^-53
(Ogita, Rump and Oishi, Accurate sum and dot product, SIAM J. Sci. Comput. 26, 2005); twice the first is allowed."""

from __future__ import annotations

import math

import numpy as np
import pytest

from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu


def z_only(n, W):
    x, z = np.zeros((n, W), np.uint64), np.zeros((n, W), np.uint64)
    z[:, 0] = np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15) & np.uint64((1 << 50) - 1)
    return x, z


@pytest.mark.parametrize("num_qubits", [50, 90])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [2, 300, 5_000, 700_000])
def test_error_of_a_sum_rounded_once(num_qubits, dtype, n):
    rng = np.random.default_rng([num_qubits, n])
    x, z = z_only(n, 1 if num_qubits <= 64 else 2)
    for cancel in (False, True):
        c = rng.standard_normal(n)
        if cancel:  # sixteen orders of magnitude, and all but a few of the terms against one another
            c *= 10.0 ** rng.uniform(-8, 8, n)
            c[n // 2:n // 2 * 2] = -c[: n // 2]
            c[:3] *= 0.5
            c = rng.permutation(c)
        c = c.astype(dtype)
        c[c == 0] = 1
        g = upload(num_qubits, x, z, c)
        got = g.expectation("z+")
        g.free()
        want = math.fsum(c.astype(np.float64))
        u = 2.0 ** -53
        assert abs(got - want) <= 2 * u * abs(want) + (n * u) ** 2 * float(np.abs(c.astype(np.float64)).sum())


@pytest.mark.parametrize("special,want", [([math.inf], math.inf), ([-math.inf], -math.inf), ([math.nan], math.nan),
                                          ([math.inf, -math.inf], math.nan), ([1.7e308, 1.7e308, 1.7e308], math.inf)])
@pytest.mark.parametrize("n", [3, 20_000])
def test_numbers_that_are_not_finite(n, special, want):
    x, z = z_only(n, 1)
    c = np.full(n, 1e-3)
    c[np.linspace(0, n - 1, len(special)).astype(int)] = special
    g = upload(50, x, z, c)
    got = g.expectation("z+")
    g.free()
    assert got == want or (math.isnan(got) and math.isnan(want))
