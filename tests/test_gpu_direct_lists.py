"""The direct pass where its workgroups and contact lists change shape: i-blocks
of eight one short and one over, the change from 16 to 8 wavefronts at 2,048
particles, and clumps in which every pair touches, so that every list is worked
off many times over.  Against the FP64 oracle at the parity bound."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4
from parity import COND_TOL, force_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nfe,side", [(7, 3, 1.5), (9, 8, 1.5), (63, 1, 3.0), (129, 64, 0.5), (700, 201, 0.55),
                                        (1201, 1200, 0.55), (2048, 700, 12.0), (2049, 64, 12.0), (2300, 900, 2.5)])
def test_direct_lists(gpu, oracle, n, nfe, side):
    rng = np.random.default_rng(n)
    pos, vel = f4(n), f4(n)
    pos[:, :3] = rng.uniform(0.0, side, (n, 3))
    vel[:, :3] = 40.0 * pos[:, :3]  # receding from about r = 0.16 on
    fc = gpu.make_impact(10, 0)[2]
    fc.NFe = nfe
    print(f"n={n} nfe={nfe} side={side}", flush=True)
    gpu.call("gi_set_tiling", 8, 3, 0, 0, 0)
    try:
        P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel), gpu.DeviceArray(n, f4(n))
        gpu.force_collision(P, V, F, n, fc)
        gpu.sync()
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
    F64, cond, near = oracle.force_collision_f64(pos, vel, fc)
    met = force_metrics(F.download(), F64, cond, near)
    print(met)
    assert met["near_threshold"] <= n // 4  # each row has up to n pairs in contact, any of which may lie at a threshold
    assert met["cond_max"] <= COND_TOL
