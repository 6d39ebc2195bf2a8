"""PP_CHECK_INVARIANTS=1 over a sum that grows in place through refinements, as it does from 2^18 terms on: a refinement's
second halves start where the first ones end, which is no violation, and the checked run gives what the unchecked gives."""

from __future__ import annotations

import numpy as np
import pytest

from paulistrings_amd import Circuit, truncation
from test_gpu_scarce_memory import spread_terms
from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu


def test_checked_growth_in_place(monkeypatch):
    circ = Circuit(50)
    for q in range(5):
        circ.rx(0.2, q)
        circ.rzz(0.1, q, q + 1)
    out = []
    for checked in ("0", "1"):
        monkeypatch.setenv("PP_CHECK_INVARIANTS", checked)
        g = upload(50, *spread_terms(300_000, 50, np.float64))
        bits = g.bucket_bits()[1]
        g.propagate(circ, truncation.coeff(1e-2), "forward")
        assert g.bucket_bits()[1] > bits
        for ch in circ.channels():
            g.apply_rotation(ch, policy=truncation.coeff(1e-1))
        out.append(g.to_host())
        g.free()
    a, b = out
    assert np.array_equal(a._x, b._x) and np.array_equal(a._z, b._z) and np.array_equal(a._c, b._c)
