"""Steps enqueued together: the sum kernel moves each particle and leaves the
next step's padded copy.  Bitwise against the same steps enqueued one call at a
time (force, then move), where the copy is made anew and the move is a kernel
of its own: the arithmetic and its order are the same."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu

TILINGS = [(4, 2, 128, 0, 64), (8, 4, 64, 0, 64), (1, 2, 64, 0, 64), (4, 0, 128, 0, 64)]  # the last has no fused move


def _state(n):
    rng = np.random.default_rng(n)
    pos, vel = f4(n), f4(n)
    pos[:, :3] = rng.uniform(-9.0, 9.0, (n, 3))
    pos[:, 3] = rng.uniform(0.0, 1.0, n)
    vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    return pos, vel


def _same(gpu, n, pos, vel, together, one):
    got = []
    for go in (together, one):
        P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel), gpu.DeviceArray(n, f4(n))
        go(P, V, F)
        gpu.sync()
        got.append([a.download() for a in (P, V, F)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert np.isfinite(got[0][0]).all() and not np.array_equal(got[0][0], pos)


@pytest.mark.parametrize("tiling", TILINGS)
@pytest.mark.parametrize("n,nfe", [(65, 1), (257, 256), (1500, 0), (2049, 700)])
def test_impact_steps(gpu, n, nfe, tiling):
    pos, vel = _state(n)
    fc, mc = gpu.make_impact(10, 0)[2:4]
    fc.NFe = mc.NFe = nfe
    print(f"n={n} nfe={nfe} {tiling}", flush=True)
    gpu.call("gi_set_tiling", *tiling)
    try:

        def one(P, V, F):
            for _ in range(17):
                gpu.force_collision(P, V, F, n, fc)
                gpu.move_collision(P, V, F, n, mc)

        _same(gpu, n, pos, vel, lambda P, V, F: gpu.impact_steps(P, V, F, n, fc, mc, 17), one)
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)


# the borders of the move need not be those of the force, nor in order
@pytest.mark.parametrize("tiling", TILINGS)
@pytest.mark.parametrize("n,b,mb", [
    (257, (1, 130, 131), (1, 130, 131)),
    (1500, (300, 700, 900), (300, 700, 900)),
    (1500, (0, 700, 1500), (900, 300, 1200)),
    (1111, (64, 512, 512), (700, 900, 200)),
])
def test_separate_steps(gpu, n, b, mb, tiling):
    pos, vel = _state(n)
    fs, ms = gpu.separate_constants(gpu.units(gpu.generator_setup_defaults(n)))
    fs.boarder1, fs.boarder2, fs.boarder3 = b
    ms.boarder1, ms.boarder2, ms.boarder3 = mb
    print(f"n={n} {b} {mb} {tiling}", flush=True)
    gpu.call("gi_set_tiling", *tiling)
    try:

        def one(P, V, F):
            for _ in range(9):
                gpu.force_separate(P, V, F, n, fs)
                gpu.move_damped_separate(P, V, F, n, ms, 6.0, 3.0)

        def together(P, V, F):
            gpu.call("gi_separate_steps", P.ptr, V.ptr, F.ptr, n, C.byref(fs), C.byref(ms), C.c_float(6.0),
                     C.c_float(3.0), 9, None)

        _same(gpu, n, pos, vel, together, one)
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
