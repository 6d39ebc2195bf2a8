"""PP_IN_PLACE_MIN_ROWS=0 has every layer of a propagation run in place, small sums' too.  The profile shows it: an in-place
layer is timed as its first launch and, when pairs are left for it, its redo launch, and counts the rows it read exactly; a
queued layer is one launch, counted at its bound.  Sums grown from two terms, so that pairs without room are redone."""

from __future__ import annotations

import numpy as np
import pytest

import pp_oracle as po
from paulistrings_amd import Circuit, PauliSum, truncation
from test_gpu_parity import oracle_policy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_qubits", [40, 90])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_every_layer_runs_in_place(monkeypatch, num_qubits, dtype):
    monkeypatch.setenv("PP_IN_PLACE_MIN_ROWS", "0")
    rng = np.random.default_rng(5)
    circ = Circuit(num_qubits)
    for _ in range(110):
        a, b = sorted(int(v) for v in rng.choice(40, 2, replace=False))
        p = str(rng.choice(["ZZ", "XX", "YZ", "X", "Y"]))
        circ.pauli_rotation(p, [a] if len(p) == 1 else [a, b], float(rng.uniform(0.3, 1.2)))
    W = 1 if num_qubits <= 64 else 2
    x, z = np.zeros((2, W), np.uint64), np.zeros((2, W), np.uint64)
    x[:, 0], z[0, 0] = (1 << 3, 1 << 11), 1 << 7
    c = np.array([1.0, -0.5], dtype)
    policy = truncation.coeff(1e-4) & truncation.weight(10)
    g = PauliSum(num_qubits, x, z, c, dtype=dtype).to_device(0)
    try:
        g.ctx.profile_enable(True)
        stats = g.propagate_with_stats(circ, policy, "forward")
        launches, _, rows_in, _ = g.ctx.profile_read()
        g.ctx.profile_enable(False)
        assert launches > len(circ.channels())  # some with a redo launch
        assert rows_in == sum(stats.terms_in)
        assert not any(v for k, v in g.check_layout().items() if k != "unscanned")
        h = g.to_host()
    finally:
        g.ctx.profile_enable(False)
        g.free()
    o = po.OracleSum(num_qubits, x, z, c)
    lens = o.propagate(circ.channels(), "forward", oracle_policy(eps=1e-4, max_weight=10))
    ox, oz, oc, _ = o.export()
    assert [int(v) for v in lens] == stats.terms_out and max(stats.terms_out) > 10_000
    assert np.array_equal(h._x, ox) and np.array_equal(h._z, oz) and np.array_equal(h._c, oc)
