"""gi_plan_info's workgroups of the direct pass: eight i-particles each,
whatever the block table's granularity."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r,n,workgroups", [(8, 2048, 256), (4, 2048, 256), (1, 2048, 256), (8, 2049, 257),
                                            (4, 2049, 258), (1, 2049, 264)])
def test_workgroups(gpu, r, n, workgroups):
    pos = f4(n)
    pos[:, 0] = 2.0 * np.arange(n)
    P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, f4(n)), gpu.DeviceArray(n, f4(n))
    fc = gpu.make_impact(10, 0)[2]
    fc.NFe = n // 4
    gpu.call("gi_set_tiling", r, 3, 0, 0, 0)
    try:
        gpu.force_collision(P, V, F, n, fc)
        gpu.sync()
        info = gpu.plan_info()
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
    assert info["kernel"] == "k_direct" and info["pair_tasks"] == workgroups
