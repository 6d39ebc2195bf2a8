"""A captured layer holds the tile sums of its output's offset scan as well as its columns: a download at a reference
bucketing far finer than the device's leaves them where they are, and a replay is refused on the host once another call has
moved them (a class pass scans its own, many more, buckets; two bring the output back to the column set it had)."""

from __future__ import annotations

import numpy as np
import pytest

from paulistrings_amd import Circuit, _native, tables, truncation
from test_gpu_scarce_memory import spread_terms
from test_gpu_transfer import upload

pytestmark = pytest.mark.gpu


def captured(n=1 << 20):
    x, z, c = spread_terms(n, 50, np.float32)
    src = upload(50, x, z, c)
    assert src.bucket_bits()[1] == 12  # more buckets than one tile of the scan holds
    while src.bucket_bits()[0] < 16:
        assert _native.lib().pp_sum_refine(src._h) == 0
    dst = src.clone()
    ch = Circuit(50).rzz(0.7, 4, 5).channels()
    src.apply_rotation_to(dst, ch, policy=truncation.coeff(1e-4))
    assert len(dst) > n
    with src.ctx.capture() as cap:
        src.apply_rotation_to(dst, ch, policy=truncation.coeff(1e-4))
    return src, dst, cap


def test_downloads_between_replays():
    src, dst, cap = captured()
    others = []
    try:
        want = None
        for rep in range(3):
            print(f"[gpu case] graph replay {rep} after a download", flush=True)
            cap.graph.launch()
            got = dst.to_host()
            want = want or got
            assert np.array_equal(got._x, want._x) and np.array_equal(got._z, want._z)
            assert np.array_equal(got._c, want._c)
            others.append(src.clone())  # takes what memory the download gave back
    finally:
        cap.graph.free()
        for g in [src, dst] + others:
            g.free()


def test_a_replay_is_refused_once_the_scan_s_scratch_moved():
    src, dst, cap = captured()
    try:
        cap.graph.launch()
        rng = np.random.default_rng(3)
        h = rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4))
        w, v = np.linalg.eigh(h + h.conj().T)
        table = tables.unitary_table((v * np.exp(-0.002j * w)) @ v.conj().T, [3, 17], np.float32)
        for _ in range(2):
            dst.apply_table(table, truncation.coeff(0.5))
        with pytest.raises(Exception, match="changed since the capture"):
            cap.graph.launch()
    finally:
        cap.graph.free()
        src.free()
        dst.free()
