"""The Earth / Moon finder at the edges of its workgroups' runs: one to a few
elements, 320 elements (united in LDS) and 1,024 (sizes counted together) one
less and one more, mostly one group and mostly loners.  Whole numbers equal
the oracle's, the FP64 sums its FP64 twin's to 1e-9."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import f4
from test_gpu_earth_moon import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density", [1.2, 0.08])
@pytest.mark.parametrize("n", [1, 2, 63, 319, 320, 321, 511, 512, 513, 641, 1023, 1025, 6001])
def test_runs_and_loners(gpu, oracle, n, density):
    rng = np.random.default_rng(n)
    pos, vel = f4(n), f4(n)
    pos[:, :3] = rng.uniform(0.0, (n / density) ** (1.0 / 3.0), (n, 3))
    vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    print(f"n={n} density={density}", flush=True)
    _check(gpu, oracle, pos, vel, n // 5, n // 10, n // 2, 2.364458)
