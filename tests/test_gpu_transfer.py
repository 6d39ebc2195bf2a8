"""Uploads bucketed and downloads sorted on the device, at the sizes where their paths change: the first size that the
device buckets, reference buckets at the edges of the sort's power-of-two sizes, either bucketing the finer one, and the
forms the host still takes (device buckets too long to order by counting, a bucket past the LDS, bucketings too far
apart).  Every download has to equal the canonical order computed in numpy from the hash rows, bit for bit."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from paulistrings_amd import DEFAULT_HASH_SEED, PauliSum, _native, circuits
from test_gpu_parity import random_sum

pytestmark = pytest.mark.gpu


def buckets(num_qubits, x, z, bits):
    W = x.shape[1]
    rx, rz = np.zeros((31, W), np.uint64), np.zeros((31, W), np.uint64)
    _native.lib().pp_hash_rows(num_qubits, ctypes.c_uint64(DEFAULT_HASH_SEED), W, rx.ctypes.data, rz.ctypes.data)
    b = np.zeros(len(x), np.uint64)
    for r in range(bits):
        ones = np.bitwise_count((x & rx[r]) ^ (z & rz[r])).sum(axis=1)
        b |= (ones.astype(np.uint64) & np.uint64(1)) << np.uint64(r)
    return b


def canonical(num_qubits, x, z, c, bits):
    cols = [z[:, w] for w in reversed(range(z.shape[1]))] + [x[:, w] for w in reversed(range(x.shape[1]))]
    order = np.lexsort(cols + [buckets(num_qubits, x, z, bits)])
    return x[order], z[order], c[order]


def distinct(rng, n, num_qubits, dtype, density=0.3):
    x, z, c = random_sum(rng, n + n // 8 + 64, num_qubits, density, dtype)
    _, at = np.unique(np.concatenate([x, z], axis=1), axis=0, return_index=True)
    at = rng.permutation(at)[:n]
    assert len(at) == n
    return x[at], z[at], c[at]


def upload(num_qubits, x, z, c):
    s = PauliSum.__new__(PauliSum)
    s.num_qubits, s.width, s.hash_seed = num_qubits, circuits.width_for(num_qubits), DEFAULT_HASH_SEED
    s._x, s._z, s._c = x, z, c
    return s.to_device(0)


def check(g, num_qubits, x, z, c):
    assert all(v == 0 for k, v in g.check_layout().items() if k != "unscanned")
    h = g.to_host()
    ex, ez, ec = canonical(num_qubits, x, z, c, g.bucket_bits()[0])
    assert np.array_equal(h._x, ex) and np.array_equal(h._z, ez) and np.array_equal(h._c, ec)


@pytest.mark.parametrize("num_qubits", [40, 64, 100, 128])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, (1 << 13) - 1, 1 << 13, (1 << 13) + 1, 70_001])
def test_round_trip(num_qubits, dtype, n):
    rng = np.random.default_rng([n, num_qubits])
    x, z, c = distinct(rng, n, num_qubits, dtype)
    zero = rng.random(n) < 0.1 if n > 1 else np.zeros(n, bool)
    c[zero] = 0.0
    c[0] = -3.0
    zero[0] = False
    g = upload(num_qubits, x, z, c)
    try:
        assert len(g) == int((~zero).sum())
        check(g, num_qubits, x[~zero], z[~zero], c[~zero])
    finally:
        g.free()


@pytest.mark.parametrize("num_qubits", [50, 127])
def test_bucketings_apart_and_forms_the_host_takes(num_qubits):
    rng = np.random.default_rng(num_qubits)
    # four device buckets of about 4096 terms each: too long to be ordered by counting
    x, z, c = distinct(rng, 1 << 18, num_qubits, np.float64)
    keep = (buckets(num_qubits, x, z, 4) == 0).nonzero()[0][: 1 << 13]
    x, z, c = x[keep], z[keep], c[keep]
    g = upload(num_qubits, x, z, c)
    check(g, num_qubits, x, z, c)
    g.free()
    # reference buckets of several device buckets up to longer than the sort's LDS, and up to 512 in a device bucket
    x, z, c = distinct(rng, 50_000, num_qubits, np.float64)
    g = upload(num_qubits, x, z, c)
    lib = _native.lib()
    bits = g.bucket_bits()[0]
    for want in (bits - 1, bits - 2, bits - 3, 0):
        assert lib.pp_sum_coarsen_to(g._h, want) == 0
        check(g, num_qubits, x, z, c)
    while g.bucket_bits()[0] <= g.bucket_bits()[1] + 8:
        assert lib.pp_sum_refine(g._h) == 0
        check(g, num_qubits, x, z, c)
    g.free()
