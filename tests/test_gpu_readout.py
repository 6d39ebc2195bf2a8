"""Read-outs in product states against math.fsum over the host's terms: uniform and mixed axes (each first-word test of the
device's sieve, and qubits with no axis), signs, sums in which no term, few or every term counts, from the empty sum to
more buckets than workgroups.  The device adds float64 values in another order: within 1e-12 of the sum of magnitudes."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest

from paulistrings_amd import _native, circuits
from test_gpu_transfer import distinct, upload

pytestmark = pytest.mark.gpu


def live_words(num_qubits):
    W = circuits.width_for(num_qubits)
    return np.array([(1 << min(64, num_qubits - 64 * w)) - 1 for w in range(W)], np.uint64)


def expected(x, z, c, ax, az, neg):
    sup = x | z
    match = ((x == (sup & ax)) & (z == (sup & az))).all(axis=1)
    sign = np.where(np.bitwise_count(sup & neg).sum(axis=1) % 2 == 1, -1.0, 1.0)
    v = (c.astype(np.float64) * sign)[match]
    return math.fsum(v), float(np.abs(v).sum()), int(match.sum())


@pytest.mark.parametrize("num_qubits,dtype", [(1, np.float64), (30, np.float64), (64, np.float32), (65, np.float32),
                                              (127, np.float64), (128, np.float64)])
@pytest.mark.parametrize("n", [0, 1, 3, 700, 20_000, 700_000])
def test_axes_and_signs(num_qubits, dtype, n):
    rng = np.random.default_rng([num_qubits, n])
    live = live_words(num_qubits)
    W = len(live)

    def word_pattern():
        return rng.integers(0, 1 << 63, W, dtype=np.uint64) * np.uint64(2) & live

    states = [(live, live * 0, live * 0), (live, live, live), (live * 0, live, live),
              (live * 0, live * 0, live * 0)]  # x+, y-, z-, no axis (the identity alone counts)
    for _ in range(3):
        ax, az = word_pattern(), word_pattern()
        states.append((ax, az, word_pattern()))
    n = min(n, 4 ** num_qubits)
    if n == 0:
        x, z, c = np.zeros((0, W), np.uint64), np.zeros((0, W), np.uint64), np.zeros(0, dtype)
    elif num_qubits == 1:
        x, z = np.array([[0], [1], [0], [1]], np.uint64)[:n], np.array([[0], [0], [1], [1]], np.uint64)[:n]
        c = rng.standard_normal(n).astype(dtype)
    else:
        x, z, c = distinct(rng, n, num_qubits, dtype)
        for k in range(0, n - 10, 3):  # a third of the terms match one of the states
            ax, az, _ = states[k % len(states)]
            on = rng.integers(0, 1 << 63, W, dtype=np.uint64)
            x[k], z[k] = on & ax, on & az
        _, at = np.unique(np.concatenate([x, z], axis=1), axis=0, return_index=True)
        x, z, c = x[at], z[at], c[at]
    g = upload(num_qubits, x, z, c)
    try:
        for ax, az, neg in states:
            want, scale, _ = expected(x, z, c, ax, az, neg)
            out = ctypes.c_double()
            arrays = [np.ascontiguousarray(a) for a in (ax, az, neg)]
            st = _native.lib().pp_expectation_product(g._h, *(a.ctypes.data for a in arrays), ctypes.byref(out))
            assert st == 0
            assert abs(out.value - want) <= 1e-12 * scale
    finally:
        g.free()
