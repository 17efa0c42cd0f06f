"""The contact grid where its buckets are not a handful: every particle in one
cell, cells that share buckets (64 buckets for a cloud many cells wide), one
particle; evaluated twice, as each grid leaves the counts for the next.
Against the FP64 oracle at the conditioned bound."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4
from parity import COND_TOL, force_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walk", [1, 9])
@pytest.mark.parametrize("n,nfe,side", [(1, 1, 1.0), (64, 20, 40.0), (65, 20, 5.0), (900, 300, 0.55), (1025, 1, 9.0),
                                        (3000, 1000, 14.0)])
def test_grid_buckets(gpu, oracle, n, nfe, side, walk):
    rng = np.random.default_rng(n)
    pos, vel = f4(n), f4(n)
    pos[:, :3] = rng.uniform(-0.5 * side, 0.5 * side, (n, 3)) + 0.31
    vel[:, :3] = 40.0 * pos[:, :3]  # receding from about r = 0.16 on
    fc = gpu.make_impact(10, 0)[2]
    fc.NFe = nfe
    print(f"n={n} nfe={nfe} side={side} walk={walk}", flush=True)
    F64, cond, near = oracle.force_collision_f64(pos, vel, fc)
    P, V = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel)
    gpu.call("gi_set_tiling", 4, 2, 256, 0, 64)
    gpu.call("gi_set_contact_walk", walk)
    try:
        out = []
        for _ in range(2):
            F = gpu.DeviceArray(n, f4(n))
            gpu.force_collision(P, V, F, n, fc)
            gpu.sync()
            out.append(F.download())
    finally:
        gpu.call("gi_set_contact_walk", 0)
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
    assert np.array_equal(out[0], out[1])
    if n == 1:
        assert np.all(out[0] == 0.0)
        return
    met = force_metrics(out[0], F64, cond, near)
    print(met)
    assert met["near_threshold"] <= n // 4  # each row has up to n pairs in contact, any of which may lie at a threshold
    assert met["cond_max"] <= COND_TOL
