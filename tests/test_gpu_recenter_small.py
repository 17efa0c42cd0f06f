"""The float recentring on either side of the size from which its sums are
taken in runs: bitwise the oracle's sequential sums, and for few particles no
more launches than sums and shift."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import f4
from test_gpu_recenter_runs import COM, MFE, VEL, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["oscillating", "binades", "ties", "nonfinite"])
@pytest.mark.parametrize("n", [2, 64, 65, 1023, 2048, 2049, 2111, 2112, 2113, 3071])
def test_bitwise_the_sequential_sum(gpu, oracle, kind, n):
    pos, vel = _state(kind, n, np.random.default_rng([n, len(kind)]))
    nfe = n // 3
    print(f"{kind} n={n}", flush=True)
    P, V = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel)
    gpu.recenter_float(P, V, n, nfe, MFE, 1.0, COM, VEL)
    po, vo = oracle.recenter_f32(pos, vel, nfe, MFE, 1.0, COM, VEL)
    assert np.array_equal(P.download(), po, equal_nan=True)
    assert np.array_equal(V.download(), vo, equal_nan=True)


@pytest.mark.parametrize("n,launches", [(40, 2), (512, 2), (2048, 2), (2049, 5)])
def test_launches(gpu, n, launches):
    lib = gpu.load()  # its HIP runtime's functions are found through it
    P, V = gpu.DeviceArray(n, f4(n)), gpu.DeviceArray(n, f4(n))
    gpu.recenter_float(P, V, n, 1, MFE, 1.0, COM, VEL)  # the scratch is made
    gpu.sync()
    st, graph, nodes = C.c_void_p(), C.c_void_p(), C.c_size_t(0)
    gpu.call("gi_stream_create", C.byref(st))
    assert lib.hipStreamBeginCapture(st, 0) == 0
    gpu.recenter_float(P, V, n, 1, MFE, 1.0, COM, VEL, stream=st.value)
    assert lib.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert lib.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0
    assert lib.hipGraphDestroy(graph) == 0
    gpu.call("gi_stream_destroy", st)
    assert nodes.value == launches
