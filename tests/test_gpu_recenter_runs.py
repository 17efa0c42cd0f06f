"""The float recentring's sums taken in runs from guessed starts: bitwise the
reference's sequential float sums (the oracle's) whatever the guesses are
worth -- window and run edges, sums that oscillate through zero, terms over
many binades, all zero, tie-heavy and non-finite values."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu

MFE = 2.364458
COM, VEL = (0.125, -0.25, 2.0), (0.0, 0.001, -0.002)


def _state(kind, n, rng):
    pos, vel = f4(n), f4(n)
    if kind == "oscillating":  # rows of a lattice: each crosses zero
        pos[:, :3] = (np.arange(3 * n).reshape(n, 3) % 61 - 30).astype(np.float32) + rng.normal(0, 0.1, (n, 3))
        vel[:, :3] = np.where(np.arange(n)[:, None] % 2 == 0, 1.0, -1.0) * rng.uniform(0.5, 1.0, (n, 3))
    elif kind == "binades":
        pos[:, :3] = rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(-9, 9, (n, 3))
        vel[:, :3] = rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(-40, -30, (n, 3))
    elif kind == "ties":  # multiples of a quarter: sums tie at large binades; one velocity is zero throughout
        pos[:, :3] = rng.integers(-(1 << 22), 1 << 22, (n, 3)) * np.float32(0.25)
        vel[:, 0] = rng.integers(1, 4, n) * np.float32(0.5)
        vel[:, 1] = np.float32(1 << 24)
        vel[n // 2, 1] = 1.0
    elif kind == "nonfinite":
        pos[:, :3] = rng.normal(0, 1, (n, 3))
        vel[:, :3] = rng.normal(0, 1, (n, 3))
        pos[n // 3, 0], pos[n // 2, 1], vel[n // 4, 2] = np.nan, np.inf, -np.inf
    return pos, vel


@pytest.mark.parametrize("kind", ["oscillating", "binades", "ties", "nonfinite"])
@pytest.mark.parametrize("n", [1, 63, 127, 128, 129, 2047, 4097, 40001, 131073])
def test_runs_are_bitwise_the_sequential_sum(gpu, oracle, kind, n):
    rng = np.random.default_rng([n, len(kind)])
    pos, vel = _state(kind, n, rng)
    nfe = n // 3
    print(f"{kind} n={n}", flush=True)
    P, V = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel)
    gpu.recenter_float(P, V, n, nfe, MFE, 1.0, COM, VEL)
    po, vo = oracle.recenter_f32(pos, vel, nfe, MFE, 1.0, COM, VEL)
    assert np.array_equal(P.download(), po, equal_nan=True)
    assert np.array_equal(V.download(), vo, equal_nan=True)
