"""Many training steps against the same steps taken on the host: the device's own shuffle replayed (splitmix64 and
Fisher-Yates), each batch's gradient from pp_model_gradient at the host's parameters, and Adam in float32 numpy.  Nonzero
moments, the bf16 copies that a step leaves for the next, a last batch that is shorter, several epochs' samples.  Both
sides round every operation to float32 once, in the same order, so parameters are equal but for the powers of the moments'
decays, which both take from the C library: 1e-6 a step is allowed, where a step itself moves them by about 1e-3."""

from __future__ import annotations

import ctypes
import sys

import numpy as np
import pytest

from paulistrings_amd import learned as PL
from test_gpu_learned import samples

pytestmark = pytest.mark.gpu

F = np.float32
powf = ctypes.CDLL("libm.so.6").powf
powf.argtypes, powf.restype = [ctypes.c_float, ctypes.c_float], ctypes.c_float


def shuffles(n, seed):
    """The order of the samples in each epoch."""
    state, order, mask = seed, list(range(n)), (1 << 64) - 1
    while True:
        for i in range(n - 1, 0, -1):
            state = (state + 0x9E3779B97F4A7C15) & mask
            v = state
            v = ((v ^ (v >> 30)) * 0xBF58476D1CE4E5B9) & mask
            v = ((v ^ (v >> 27)) * 0x94D049BB133111EB) & mask
            j = (v ^ (v >> 31)) % (i + 1)
            order[i], order[j] = order[j], order[i]
        yield np.array(order)


def adam(p, m, v, g, step, lr):
    b1, b2 = F(0.9), F(0.999)
    m = b1 * m + (F(1) - b1) * g
    v = b2 * v + (F(1) - b2) * g * g
    c1, c2 = F(1) - F(powf(b1, step)), F(1) - F(powf(b2, step))
    return p - F(lr) * (m / c1) / (np.sqrt(v / c2) + F(1e-8)), m, v


@pytest.mark.parametrize("n,batch,epochs", [(1, 64, 4), (100, 128, 4), (200, 64, 2), (1000, 384, 3), (1500, 1024, 2),
                                            (2048, 512, 2)])
def test_steps_and_epochs(n, batch, epochs):
    print(f"[gpu case] mlp training steps n={n} batch={batch} epochs={epochs}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng([n, batch])
    groups = PL.lattice_groups(8, 8)
    x, z, c, rem = samples(rng, n)
    labels = rng.standard_normal(n).astype(np.float32)
    device = PL.Model(groups, depth_scale=40.0, seed=11)
    host = PL.Model(groups, depth_scale=40.0, seed=11)
    p = device.get_params()
    got = device.train(x, z, c, rem, labels, epochs=epochs, batch=batch, lr=1e-3, seed=3)
    m, v, step = np.zeros_like(p), np.zeros_like(p), 0
    start = p
    epoch_orders = shuffles(n, 3)
    for _ in range(epochs):
        order, squares = next(epoch_orders), 0.0
        for at in range(0, n, batch):
            b = order[at:at + batch]
            host.set_params(p)
            g, loss = host.gradient(x[b], z[b], c[b], rem[b], labels[b])
            squares += loss * len(b)
            step += 1
            p, m, v = adam(p, m, v, g, step, 1e-3)
    after = device.get_params()
    device.free()
    host.free()
    assert p.dtype == np.float32 and step == epochs * -(-n // batch)
    assert np.abs(after - p).max() <= 1e-6 * step, float(np.abs(after - p).max())
    assert np.abs(after - start).max() > 1e-3  # the steps moved parameters (one sample leaves most units' alone)
    assert abs(got - squares / n) <= 1e-9 * max(1.0, got)
