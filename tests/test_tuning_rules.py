"""The rules of giant-impact_amd/csrc/gi_tuning.h on the host alone (built with
g++): on either side of each line, where both forms were timed, the faster one
(or either, where they take the same time)."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "tuning_rules"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(REPO / "giant-impact_amd" / "csrc"),
                    str(REPO / "tests" / "cpp" / "tuning_rules.cpp"), "-ldl", "-o", str(exe)], check=True)

    def run(*a):
        return int(subprocess.run([str(exe), *map(str, a)], capture_output=True, text=True, check=True).stdout)

    return run


# (simulations, particles of each): one simulation; the step of several was
# timed with one lane and with nine
@pytest.mark.parametrize("sims,n,lanes", [
    (1, 13000, 9), (1, 49152, 9), (1, 49153, 1), (1, 65536, 1),
    (8, 1100, 9), (64, 2048, 9), (160, 2048, 9), (256, 2048, 1), (384, 2048, 1),
    (96, 3000, 9), (192, 3000, 1), (64, 4096, 9), (128, 4096, 1), (256, 4096, 1),
    (32, 6000, 9), (48, 6000, 1), (64, 6000, 1), (16, 8000, 9), (32, 8000, 1), (48, 8000, 1),
    (8, 12000, 9), (16, 12000, 1), (64, 12000, 1),
])
def test_contact_walk(rule, sims, n, lanes):
    assert rule("walk", sims, n) == lanes


# (particles, the engine's length, j per piece): the longest length, or within
# 1-2% of the fastest, for a full GPU of such simulations
@pytest.mark.parametrize("n,full,length", [
    (1, 768, 64), (2048, 768, 64), (3072, 768, 64), (3073, 768, 128), (4096, 768, 128), (5120, 768, 128),
    (6000, 768, 192), (7000, 768, 192), (8000, 768, 256), (10000, 768, 256), (12000, 768, 256), (16384, 768, 256),
    (16385, 768, 384), (20000, 768, 448), (24576, 768, 512), (24577, 768, 768), (65536, 768, 768),
    (65536, 4096, 2048), (8000, 128, 128), (20000, 64, 64),
])
def test_batched_piece(rule, n, full, length):
    assert rule("piece", n, full) == length


# where the class above or below would take single calls longer than the forms
# that had these sizes before them
@pytest.mark.parametrize("n,R,variant,length", [
    (12289, 4, 2, 128), (24576, 4, 2, 128), (24577, 4, 2, 256), (25300, 4, 2, 256), (27600, 4, 2, 256),
    (33792, 4, 2, 256), (33793, 8, 4, 128), (49152, 8, 4, 128), (49153, 8, 4, 256),
])
def test_mid_size_rows(gi, n, R, variant, length):
    t = gi.tiling_for(n)
    assert (t["r"], t["variant"], t["chunk_len"]) == (R, variant, length)
