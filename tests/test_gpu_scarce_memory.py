"""Calls that take more device memory than they need when there is plenty of it, with most of the device's memory taken by
another owner: they have to fall back to what they cannot do without, with the same result."""

from __future__ import annotations

import contextlib

import numpy as np
import pytest

from paulistrings_amd import tables, truncation
from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu

MB = 1 << 20


@contextlib.contextmanager
def device_memory_left(megabytes):
    torch = pytest.importorskip("torch")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    taken = []
    try:
        for _ in range(10):  # memory just freed may be reported late
            more = torch.cuda.mem_get_info()[0] - megabytes * MB
            if more <= 16 * MB:
                break
            taken.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        assert abs(torch.cuda.mem_get_info()[0] - megabytes * MB) <= 32 * MB
        yield
    finally:
        taken.clear()
        torch.cuda.empty_cache()


def spread_terms(n, num_qubits, dtype):
    """n distinct one-word terms (an odd multiplier permutes the x words)."""
    mask = np.uint64((1 << num_qubits) - 1)
    i = np.arange(n, dtype=np.uint64)
    x = (i * np.uint64(0x9E3779B97F4A7C15)) & mask
    z = (i * np.uint64(0xD1B54A32D192ED03) >> np.uint64(7)) & mask
    return x.reshape(-1, 1), z.reshape(-1, 1), (1.0 + i % 1000).astype(dtype)


def test_an_upload_beside_little_free_memory():
    """2^23 terms: the columns take 275 MB, the terms as they arrive, bucketed on the device, 235 MB more."""
    x, z, c = spread_terms(1 << 23, 50, np.float32)
    g = upload(50, x, z, c)
    want = g.to_host()
    g.free()
    with device_memory_left(400):
        g = upload(50, x, z, c)
        assert len(g) == len(c)
    assert not any(v for k, v in g.check_layout().items() if k != "unscanned")
    got = g.to_host()
    g.free()
    assert np.array_equal(got._x, want._x) and np.array_equal(got._z, want._z) and np.array_equal(got._c, want._c)


@pytest.mark.parametrize("left", [1010, 790, 640, 540])
def test_a_general_table_beside_little_free_memory(left):
    """2^22 terms through a near-identity two-qubit unitary whose small outputs are dropped.  The rows it moves take 190 MB,
    the outputs are staged in room for four times the terms, 384 MB, and the columns they are placed in take 112.  With
    640 MB left the staging fits and the columns do not, with 540 half of the staging fits; twice the staging (768 MB) would
    leave no room for the columns with 1010."""
    n = 1 << 22
    x, z, c = spread_terms(n, 50, np.float32)
    rng = np.random.default_rng(3)
    h = rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4))
    w, v = np.linalg.eigh(h + h.conj().T)
    table = tables.unitary_table((v * np.exp(-0.002j * w)) @ v.conj().T, [3, 17], np.float32)
    assert table.n_deltas == 16
    c = 1.0 + c / 2000
    policy = truncation.coeff(0.5)
    g = upload(50, x, z, c)
    g.apply_table(table, policy)
    want = g.to_host()
    g.free()
    assert len(want) == n
    g = upload(50, x, z, c)
    with device_memory_left(left):
        g.apply_table(table, policy)
    assert not any(v for k, v in g.check_layout().items() if k != "unscanned")
    got = g.to_host()
    g.free()
    assert np.array_equal(got._x, want._x) and np.array_equal(got._z, want._z) and np.array_equal(got._c, want._c)


def test_columns_beside_a_selection_s_scratch():
    """A sum of 2^24 terms keeps 128 MB of scratch of its last selection, then takes a sum of 2^25: columns of 1020 MB in
    place of its 510, with 448 MB left."""
    terms = spread_terms(1 << 25, 50, np.float32)
    src, dst = upload(50, *terms), upload(50, *(a[: 1 << 24] for a in terms))
    for n in ((1 << 24) - 5, (1 << 24) - 10):  # the second starts from the boundary of the first
        dst.truncate_topn(n)
        assert len(dst) == n
    with device_memory_left(448):
        dst.copy_from(src)
        dst.ctx.sync()
    assert not any(v for k, v in dst.check_layout().items() if k != "unscanned")
    want = src.to_host()
    src.free()
    got = dst.to_host()
    dst.free()
    assert np.array_equal(got._x, want._x) and np.array_equal(got._z, want._z) and np.array_equal(got._c, want._c)
