"""Two bodies in one launch take the plan of one simulation with as many pairs:
sizes on both sides of the direct pass's line (sqrt(n1^2 + n2^2) against
12,288), where the two bodies together lie beyond it, and of the next classes.
Against the FP64 oracle at the conditioned bound."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import f4
from parity import COND_TOL, force_metrics


@pytest.mark.gpu
@pytest.mark.parametrize("n1,n2,kernel", [(8688, 8688, "k_direct"), (8690, 8689, "k_mutual"), (12288, 1, "k_mutual"),
                                          (12200, 900, "k_direct"), (20500, 20400, "k_mutual"),
                                          (24100, 24000, "k_mutual_grp")])
def test_two_bodies_by_pairs(gpu, oracle, n1, n2, kernel):
    from test_gpu_force import _generator_bodies

    pos, vel, fs, _ = _generator_bodies(gpu, n1, n2, 3)
    n = len(pos)
    print(f"n1={n1} n2={n2}", flush=True)
    P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel), gpu.DeviceArray(n, f4(n))
    gpu.force_separate(P, V, F, n, fs)
    gpu.sync()
    assert gpu.plan_info()["kernel"] == kernel
    met = force_metrics(F.download(), *oracle.force_separate_f64(pos, vel, fs))
    print(met)
    assert met["near_threshold"] <= n // 100
    assert met["cond_max"] <= COND_TOL


def test_workgroup_lists_of_every_length(gi):
    """Task lists around whole runs of 256 workgroups and the longest list that
    is dealt out: every block is still taken exactly once (host only)."""
    lib = gi.load()
    for n in list(range(256, 4000, 251)) + [9000, 12289, 15000, 20000, 21001, 27648]:
        a, b = (C.c_int * 1)(n), (C.c_int * 1)(n // 3)
        for r, v, L in ((1, 2, 64), (4, 2, 64), (4, 2, 128), (8, 4, 128), (4, 4, 64)):
            for batched in (0, 1):
                assert lib.gi_plan_check(1, a, b, r, v, C.c_longlong(L), batched) == 0, (n, r, v, L, batched)
