"""ApproxTopN's cut (whole octaves of |c|^2 from the top, the boundary octave's first terms in canonical order) against
numpy, in the forms the device's cut meets: quotas from none of the boundary octave to all but one of it, reference
buckets of one and of many device buckets, a split bucket past what one workgroup orders and reference buckets finer than
the device's (both walked on the host), one octave for all terms, NaNs and infinities; and inside a propagation, where the
retain is left to the next layer, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

import pp_oracle as po
from paulistrings_amd import Circuit, PauliSum, _native, truncation
from test_gpu_transfer import canonical, distinct, upload

pytestmark = pytest.mark.gpu


def cut(num_qubits, x, z, c, bits, n):
    x, z, c = canonical(num_qubits, x, z, c, bits)
    if len(c) <= n:
        return x, z, c
    with np.errstate(over="ignore", invalid="ignore"):
        u = c.astype(np.float64) ** 2
    nan = np.isnan(u)
    octave = np.where(nan, 2047, (u.view(np.uint64) >> np.uint64(52)).astype(np.int64) & 2047)
    hist = np.bincount(octave, minlength=2048)
    above = 0
    for o in range(2047, -1, -1):
        if above + hist[o] > n:
            break
        above += hist[o]
    stay = (octave > o) & ~nan
    boundary = ((octave == o) & ~nan).nonzero()[0]
    stay[boundary[: n - above]] = True
    return x[stay], z[stay], c[stay]


@pytest.mark.parametrize("num_qubits,dtype", [(50, np.float64), (127, np.float64), (64, np.float32), (100, np.float32)])
@pytest.mark.parametrize("values", ["normal", "octave", "special"])
@pytest.mark.parametrize("n", [900, 9_000, 60_000])
def test_cuts(num_qubits, dtype, values, n):
    rng = np.random.default_rng([num_qubits, n])
    x, z, c = distinct(rng, n, num_qubits, dtype)
    if values == "octave":
        c = (np.sign(c) * (1.01 + 0.3 * rng.random(n))).astype(dtype)  # |c|^2 in [1.02, 1.72]
    elif values == "special":
        c[rng.random(n) < 0.1] = np.nan
        c[rng.random(n) < 0.1] = np.inf
        c[rng.random(n) < 0.1] = -np.inf
    lib = _native.lib()
    base = upload(num_qubits, x, z, c)
    bits0 = base.bucket_bits()[0]
    try:
        for bits in sorted({0, bits0 - 1, bits0, bits0 + 2} & set(range(20))):
            g = base.clone()
            while g.bucket_bits()[0] < bits:
                assert lib.pp_sum_refine(g._h) == 0
            assert lib.pp_sum_coarsen_to(g._h, bits) == 0
            hx, hz, hc = x, z, c
            for k in (n - 1, n - n // 10, n // 2 + 1, n // 2, n // 7, 1):
                g.truncate_approx_topn(k)
                hx, hz, hc = cut(num_qubits, hx, hz, hc, bits, k)
                h = g.to_host()
                assert len(h) == len(hc), (bits, k)
                assert np.array_equal(h._x, hx) and np.array_equal(h._z, hz), (bits, k)
                assert np.array_equal(h._c, hc, equal_nan=True), (bits, k)
            assert all(v == 0 for key, v in g.check_layout().items() if key != "unscanned")
            g.free()
    finally:
        base.free()


@pytest.mark.parametrize("num_qubits,dtype,n", [(40, np.float64, 5_000), (100, np.float32, 5_000), (60, np.float64, 300_000)])
def test_inside_a_propagation(num_qubits, dtype, n):
    rng = np.random.default_rng(n + num_qubits)
    x, z, c = distinct(rng, n, num_qubits, dtype, density=0.1)
    circ = Circuit(num_qubits)
    for i in range(24):
        a, b = (int(v) for v in rng.choice(num_qubits, size=2, replace=False))
        if i % 5 == 4:
            circ.pauli_rotation("ZZ", [a, b], np.pi / 2)  # Clifford: a permutation step between the cuts
        elif i % 2:
            circ.pauli_rotation("ZZ", [a, b], 0.4)
        else:
            circ.rx(0.3, a)
    o = po.OracleSum(num_qubits, x, z, c)
    lens = o.propagate(circ.channels(), "heisenberg", po.coeff_policy(eps=1e-6, approx_topn=n))
    ox, oz, oc, _ = o.export()
    g = upload(num_qubits, x, z, c)
    try:
        stats = g.propagate_with_stats(circ, truncation.coeff(1e-6) & truncation.approx_topn(n), "heisenberg")
        h = g.to_host()
    finally:
        g.free()
    assert [int(v) for v in lens] == stats.terms_out
    assert np.array_equal(h._x, ox) and np.array_equal(h._z, oz) and np.array_equal(h._c, oc)
