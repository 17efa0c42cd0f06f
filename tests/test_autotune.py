"""The autotuner's candidates (host only)."""
from __future__ import annotations

import pytest

from gi_amd import autotune


@pytest.mark.parametrize("n_max,nt,ni", autotune.CLASSES)
def test_one_candidate_per_form(n_max, nt, ni):
    """No two candidates of a class run the same force: the direct pass's R
    changes its energy pass alone, so it is timed once."""
    c = autotune.candidates(n_max, nt + ni, [1, 2, 4, 8], [0], [4096, 8192], [128, 512])
    assert len(set(c)) == len(c)
    assert sum(t[1] == 3 for t in c) == (1 if n_max <= autotune.DIRECT_MAX_CLASS else 0)
    assert {t[1] for t in c} >= {0, 2, 4}
