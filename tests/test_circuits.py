"""A circuit's channels in the layout the C ABI reads."""

import numpy as np
import pytest

from paulistrings_amd import _channel_rows, circuits


def plain(circuit):
    out = np.zeros(len(circuit), circuits.CHANNEL_DTYPE)
    for i, (gx, gz, theta) in enumerate(circuit._rows):
        out["gx"][i], out["gz"][i], out["theta"][i] = gx, gz, theta
    return out


@pytest.mark.parametrize("qubits", [1, 64, 65, 128])
@pytest.mark.parametrize("kind", [int, np.int64, np.uint64])
def test_channels_hold_every_word_bit_and_angle(qubits, kind):
    c = circuits.Circuit(qubits)
    assert c.channels().dtype == circuits.CHANNEL_DTYPE and len(c.channels()) == 0
    for q in sorted({0, qubits // 2, qubits - 1}):
        for p in "XYZ":
            c.pauli_rotation(p, [kind(q)], 0.1 * q - 1.0 / 3.0)
    got = c.channels()
    assert got.flags.writeable and got.flags.c_contiguous
    assert got.tobytes() == plain(c).tobytes()
    assert _channel_rows(got).tobytes() == got.tobytes()
    assert _channel_rows(got[::2]).tobytes() == got[::2].tobytes()
    assert _channel_rows(got.reshape(-1, 1)).tobytes() == got.tobytes()
