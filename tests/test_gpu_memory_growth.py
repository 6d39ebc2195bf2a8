"""Device memory held by one sum through many passes: a working sum reset from a resident one and propagated through
refinements, and a sum replaced by its clone, again and again, have to stay at the size of the first few passes."""

from __future__ import annotations

import numpy as np
import pytest

from paulistrings_amd import Circuit, truncation
from test_gpu_scarce_memory import MB, spread_terms
from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu


def used():
    torch = pytest.importorskip("torch")
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


@pytest.mark.parametrize("layers", [2, 6])
def test_reset_and_propagate(layers):
    src = upload(50, *spread_terms(1 << 19, 50, np.float64))
    work = src.clone()
    circ = Circuit(50)
    for q in range(layers):
        circ.rx(0.7, q)
    bits = src.bucket_bits()[1]
    lens, after = set(), []
    for _ in range(14):
        work.copy_from(src)
        work.propagate(circ, truncation.coeff(1e-9), "forward")
        lens.add(len(work))
        after.append(used())
    assert len(lens) == 1 and work.bucket_bits()[1] > bits  # refined
    src.free()
    work.free()
    # a quarter more at each of eleven passes would be twelve times the columns, 40 MB and more
    assert after[-1] - min(after[2:5]) < 40 * MB, [a // MB for a in after]


def test_clones_of_clones():
    g = upload(50, *spread_terms(1 << 19, 50, np.float64))
    after = []
    for _ in range(14):
        h = g.clone()
        g.free()
        g = h
        after.append(used())
    g.free()
    assert after[-1] - min(after[2:5]) < 40 * MB, [a // MB for a in after]
