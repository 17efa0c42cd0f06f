"""The direct pass's sums where float sums of their partial results would drop
what is left after large terms cancel: across the lanes of a wavefront, along a
lane's j at sizes far above the table's, and over a batch of contact terms.

Particle 0's force from particles on the x axis, whose terms are powers of two
(r^2 a power of four), or contact terms that are exact in float: every partial
sum of like terms is exact, so the force has to be the exact sum rounded once.
Runs of at least eight consecutive particles share a term, except in the
contact test, whose runs are of four and more: terms of different size meet
only where the pass no longer adds in plain float."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4

pytestmark = pytest.mark.gpu

FAR = np.float32(1e18)  # its gravity term is zero


def _force0(gpu, pos, vel, fc, r):
    n = len(pos)
    gpu.call("gi_set_tiling", r, 3, 0, 0, 0)
    try:
        P, V, F = gpu.DeviceArray(n, pos), gpu.DeviceArray(n, vel), gpu.DeviceArray(n, f4(n))
        gpu.force_collision(P, V, F, n, fc)
        gpu.sync()
    finally:
        gpu.call("gi_set_tiling", 0, 0, 0, 0, 0)
    return F.download()[0]


def _law(gpu):
    fc = gpu.make_impact(10, 0)[2]
    fc.NFe = 0
    return fc


@pytest.mark.parametrize("r", [1, 8])
def test_one_pair_is_exact(gpu, r):
    """What the tests below rest on: the term of a pair 2^a apart is 4^-a."""
    for a in range(1, 15):
        pos = f4(2)
        pos[1, 0] = np.float32(2.0**a)
        assert _force0(gpu, pos, f4(2), _law(gpu), r)[0] == np.float32(4.0**-a)


@pytest.mark.parametrize("n", [512, 1024, 2048, 4096])
def test_lanes_of_a_wavefront(gpu, n):
    """Half rows of lanes alternate between a large term and a small one, rows
    between the two signs of the large one."""
    j = np.arange(n)
    big = j % 16 < 8
    sign = np.where(j // 16 % 2 == 0, 1.0, -1.0)
    pos = f4(n)
    pos[:, 0] = np.where(big, 2.0 * sign, 2.0**14)
    pos[0, 0] = 0.0
    pos[16, 0] = FAR  # what balances particle 0 itself
    exact = np.where(big, 0.25 * sign, 2.0**-28)
    exact[[0, 16]] = 0.0
    print(f"n={n}", flush=True)
    f = _force0(gpu, pos, f4(n), _law(gpu), 8)
    assert f[0] == np.float32(exact.sum()) and f[0] == np.float32(n * 2.0**-29)
    assert f[1] == 0.0 and f[2] == 0.0


def test_along_j(gpu):
    """Each lane takes 64 large terms, 64 small ones and 64 large ones of the
    other sign."""
    n = 3 * 64 * 512
    part = np.arange(n) // (64 * 512)
    pos = f4(n)
    pos[:, 0] = np.choose(part, [2.0, 2.0**14, -2.0])
    pos[0, 0] = 0.0
    pos[2 * 64 * 512, 0] = FAR
    print(f"n={n}", flush=True)
    f = _force0(gpu, pos, f4(n), _law(gpu), 8)
    assert f[0] == np.float32(64 * 512 * 2.0**-28)


def test_contact_batches(gpu):
    """Of each 64 j, 32 are in stiff contact, 4 in weak contact (receding),
    and the stiff ones of every other 512 pull the other way."""
    fc = _law(gpu)
    fc.KSiSi, fc.KRSiSi, fc.ShellBreakSi = 2.0**22, 0.0, 0.9
    n = 2048
    j = np.arange(n)
    lane, sign = j % 64, np.where(j // 512 % 2 == 0, 0.5, -0.5)
    stiff, weak = lane < 32, (lane >= 32) & (lane < 36)
    out = (j < 64) | ((j >= 512) & (j < 576))  # particle 0's block and the one that balances it
    pos, vel = f4(n), f4(n)
    pos[:, 0] = np.where(out, FAR, np.where(stiff, sign, np.where(weak, 0.5, FAR)))
    vel[:, 0] = np.where(weak, 100.0, 0.0)
    pos[0, 0] = 0.0
    pos[1:8, 0] = 0.0  # its neighbours in the i-block: each alone, far away
    pos[1:8, 1] = FAR * np.float32(2.0) ** np.arange(1, 8, dtype=np.float32)
    vel[:8, 0] = 0.0
    f = _force0(gpu, pos, vel, fc, 8)
    weak_in = int((weak & ~out).sum())
    assert weak_in == 120
    assert f[0] == np.float32(weak_in)  # G - KR (1 - r^2) = 1 each
