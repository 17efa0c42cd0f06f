"""Runs of steps queue in stream order behind what was enqueued before them and
ahead of what follows, without the caller waiting (on the default stream), with
a step's work on one stream or forked (the contact grid beside the mutual
pass).  Bitwise against the same calls with a wait after each."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tiling", [(1500, (8, 3, 0, 0, 0)), (40000, (4, 2, 256, 0, 64)), (3000, (8, 4, 64, 0, 64))])
def test_steps_in_stream_order(gpu, n, tiling):
    pos, vel, fc, mc, _ = gpu.make_impact(n - n // 4, n // 4, seed=5, speed_vesc=1.2)
    print(f"n={n} {tiling}", flush=True)
    got = []
    gpu.call("gi_set_tiling", *tiling)
    try:
        for wait in (True, False):
            P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel), gpu.DeviceArray(n, f4(n))
            mid, end = gpu.DeviceArray(n, f4(n)), gpu.DeviceArray(n, f4(n))
            gpu.sync()

            def then():
                if wait:
                    gpu.sync()

            for _ in range(3):
                for _ in range(3):  # work ahead of the steps
                    gpu.force_collision(P, V, F, n, fc)
                    gpu.move_collision(P, V, F, n, mc)
                    then()
                gpu.impact_steps(P, V, F, n, fc, mc, 17)
                then()
                gpu.call("gi_copy_d2d", mid.ptr, P.ptr, 16 * n, None)
                then()
                gpu.impact_steps(P, V, F, n, fc, mc, 9)
                then()
            gpu.call("gi_copy_d2d", end.ptr, P.ptr, 16 * n, None)
            gpu.call("gi_stream_sync", None)
            got.append([a.download() for a in (mid, end, V, F)])
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert np.isfinite(got[0][1]).all() and not np.array_equal(got[0][0], got[0][1])
