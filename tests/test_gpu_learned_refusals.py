"""What the learned propagation refuses, whatever the sum's size and however its layers are queued: a two-word sum, which
its network cannot score."""

from __future__ import annotations

import numpy as np
import pytest

from paulistrings_amd import Circuit, PauliSum, _native
from paulistrings_amd import learned as PL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [1, 100, 1_000_000])
@pytest.mark.parametrize("layers", [1, 12])
def test_a_two_word_sum_is_refused(keep, layers):
    circ = Circuit(100)
    for q in range(layers):
        circ.rx(0.1, q)
    x, z = np.zeros((1, 2), np.uint64), np.zeros((1, 2), np.uint64)
    z[0, 0] = 0x3FF
    m = PL.Model(PL.lattice_groups(8, 8), depth_scale=40.0, seed=1)
    g = PauliSum(100, x, z, np.ones(1)).to_device(0)
    try:
        with pytest.raises(_native.NativeError, match="one-word"):
            PL.propagate_learned(g, circ, m, keep)
        PL.propagate_learned(g, Circuit(100), m, keep)  # nothing to score
    finally:
        g.free()
        m.free()
