"""gi_recenter_float in a caller's own graph: captured at one size after calls
at a smaller one, and replayed after calls at a larger one, it is bitwise the
reference's sequential sums (the oracle's) each time."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu

MFE = 2.364458
COM, VEL = (0.125, -0.25, 2.0), (0.0, 0.001, -0.002)


def _state(n):
    rng = np.random.default_rng(n)
    pos, vel = f4(n), f4(n)
    pos[:, :3] = rng.normal(1.0, 8.0, (n, 3))
    vel[:, :3] = rng.normal(-0.1, 1.0, (n, 3))
    return pos, vel


@pytest.mark.parametrize("n0,n,n1", [(64, 3000, 65536), (500, 20001, 200000)])
def test_graph_outlives_calls_at_other_sizes(gpu, oracle, n0, n, n1):
    lib = gpu.load()  # its HIP runtime's functions are found through it

    def hip(name, *a):
        assert getattr(lib, name)(*a) == 0, name

    def eager(m):
        pos, vel = _state(m)
        P, V = gpu.DeviceArray(m, pos), gpu.DeviceArray(m, vel)
        gpu.recenter_float(P, V, m, m // 4, MFE, 1.0, COM, VEL)
        gpu.sync()
        want = oracle.recenter_f32(pos, vel, m // 4, MFE, 1.0, COM, VEL)
        assert np.array_equal(P.download(), want[0]) and np.array_equal(V.download(), want[1])

    print(f"n={n0},{n},{n1}", flush=True)
    eager(n0)
    pos, vel = _state(n)
    P, V = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel)
    gpu.sync()
    st, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    gpu.call("gi_stream_create", C.byref(st))
    hip("hipStreamBeginCapture", st, 0)
    gpu.recenter_float(P, V, n, n // 4, MFE, 1.0, COM, VEL, stream=st.value)
    hip("hipStreamEndCapture", st, C.byref(graph))
    hip("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    for k in range(3):
        if k:
            eager(n1 if k == 1 else n0)
        hip("hipGraphLaunch", run, st)
        gpu.call("gi_stream_sync", st)
        pos, vel = oracle.recenter_f32(pos, vel, n // 4, MFE, 1.0, COM, VEL)
        assert np.array_equal(P.download(), pos) and np.array_equal(V.download(), vel)
    hip("hipGraphExecDestroy", run)
    hip("hipGraphDestroy", graph)
    gpu.call("gi_stream_destroy", st)
