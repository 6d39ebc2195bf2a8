"""A general table's two ways through a class pass, a thread per row and a thread per pattern of a class, at tables that make
one output of a term, a few, or all of its class's, and at classes of one term and of many: every output's key and, within
1e-12, its coefficient as the naive layer gives them (bit for bit where each output has one source)."""

from __future__ import annotations

import numpy as np
import pytest

import ptm
from paulistrings_amd import tables, truncation
from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)
CNOT = np.array([[1, 0, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0], [0, 1, 0, 0]], float)
SWAP = np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], float)


def gate(name):
    rng = np.random.default_rng(5)
    real = np.linalg.qr(rng.standard_normal((4, 4)))[0]
    full = np.linalg.qr(rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4)))[0]
    one = np.linalg.qr(rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2)))[0]
    return {"h": (H, [4]), "one": (one, [4]), "cnot": (CNOT, [4, 5]), "swap": (SWAP, [2, 5]),
            "h x one": (np.kron(H, one), [4, 5]), "real": (real, [3, 5]), "full": (full, [4, 5])}[name]


@pytest.mark.parametrize("name", ["h", "one", "cnot", "swap", "h x one", "real", "full"])
@pytest.mark.parametrize("crowded", [False, True])
@pytest.mark.parametrize("n", [1, 16, 17, 300, 3000])
def test_outputs(name, crowded, n):
    u, qubits = gate(name)
    rng = np.random.default_rng([n, crowded])
    live = np.uint64(0x3F if crowded else (1 << 40) - 1)  # 4096 keys: a class of two qubits holds many of them
    keys = np.unique(rng.integers(0, 1 << 62, (4 * n + 64, 2), dtype=np.uint64) & live, axis=0)
    keys = keys[rng.permutation(len(keys))][:n]
    assert len(keys) == n or crowded
    x, z, c = keys[:, :1].copy(), keys[:, 1:].copy(), rng.standard_normal(len(keys))
    table = tables.unitary_table(u, qubits)
    g = upload(40, x, z, c)
    try:
        g.apply_table(table, truncation.coeff(1e-9))
        assert not any(v for k, v in g.check_layout().items() if k != "unscanned")
        h = g.to_host()
    finally:
        g.free()
    entries = [(table.deltas[e].local_delta, list(table.deltas[e].amplitude)) for e in range(table.n_deltas)]
    want = ptm.naive_table_layer({((int(a),), (int(b),)): float(v) for a, b, v in zip(x[:, 0], z[:, 0], c)}, qubits,
                                 entries, lambda kx, kz, v: abs(v) > 1e-9)
    got = {((int(a),), (int(b),)): float(v) for a, b, v in zip(h._x[:, 0], h._z[:, 0], h._c)}
    assert got.keys() == want.keys()
    one_source = name in ("cnot", "swap")
    assert all(abs(got[k] - want[k]) <= (0.0 if one_source else 1e-12) for k in want)
