"""Sums freed on another thread, as a garbage collector frees them, while this one makes and reads sums of the same context:
the pool of pinned slots that the sums' counters and answers arrive in is shared, and no slot may serve two sums."""

from __future__ import annotations

import queue
import threading

import numpy as np
import pytest

from paulistrings_amd import Circuit, PauliSum, truncation

pytestmark = pytest.mark.gpu


def test_freeing_on_another_thread():
    sources = []
    for n in (3, 40, 700):
        x = np.zeros((n, 1), np.uint64)
        z = np.arange(1, n + 1, dtype=np.uint64).reshape(-1, 1)
        sources.append(PauliSum(30, x, z, np.full(n, 1.0 / n)).to_device(0))
    circ = Circuit(30)
    for q in range(6):
        circ.rx(0.3, q)
    want = []
    for s in sources:
        g = s.clone()
        g.propagate(circ, truncation.coeff(1e-12), "forward")
        want.append((len(s), len(g), s.expectation("z+"), g.expectation("z+")))
        g.free()
    done = queue.Queue()

    def free_all():
        while (g := done.get()) is not None:
            g.free()

    worker = threading.Thread(target=free_all)
    worker.start()
    try:
        for k in range(400):
            i = k % len(sources)
            g = sources[i].clone()
            before = len(g), g.expectation("z+")
            g.propagate(circ, truncation.coeff(1e-12), "forward")
            assert (before[0], len(g), before[1], g.expectation("z+")) == want[i]
            done.put(g)
    finally:
        done.put(None)
        worker.join()
        for s in sources:
            s.free()
