"""A simulation whose contact walk takes nine lanes per particle alone and one
in a mix beyond the walk's line (about 240,000 particles): bitwise the same."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_ensemble import _ensemble_of_one

pytestmark = pytest.mark.gpu


def test_alone_and_in_a_mix_beyond_the_line(gpu):
    cfg = gpu.ensemble_configs(22, seed=8, n_range=(10600, 11400))
    pos, vel, n, fc, mc, _ = gpu.make_ensemble(cfg)
    ntot, pairs = float(n.sum()), float((n.astype(np.float64) ** 2).sum())
    assert ntot / 450000.0 + pairs / 3.0e9 > 1.0
    assert max(k / 450000.0 + k * k / 3.0e9 for k in n.astype(np.float64)) < 1.0
    print("n =", list(n), flush=True)
    P, V = gpu.DeviceArray(len(pos), pos), gpu.DeviceArray(len(pos), vel)
    ens = gpu.Ensemble(P, V, n, fc, mc)
    ens.steps(3)
    gpu.sync()
    p_all, v_all = P.download(), V.download()
    off = ens.offsets
    ens.close()
    for s in (0, 11, 21):
        a, b = off[s], off[s + 1]
        p1, v1 = _ensemble_of_one(gpu, pos[a:b], vel[a:b], fc[s], mc[s], 3)
        assert np.array_equal(p_all[a:b], p1), s
        assert np.array_equal(v_all[a:b], v1), s
