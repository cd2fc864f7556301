"""Extension by a group of 16 lanes (g3a_ext_group.h) on the CPU: its lanes as
fibers, against the oracle's banded extension, over short and long queries,
narrow bands, three gap-cost kinds and targets that return to h0
(tests/ext_group_check.cpp)."""
from __future__ import annotations

import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    out = tmp_path_factory.mktemp("ext_group") / "ext_group_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(ROOT), "-o", str(out),
                    str(ROOT / "tests" / "ext_group_check.cpp"), "-x", "c", str(ROOT / "oracle" / "oracle.c"), "-lm"],
                   check=True, capture_output=True)
    return out


@pytest.mark.parametrize("seed", [1, 2])
def test_ext_group_equals_oracle(checker, seed):
    r = subprocess.run([str(checker), "3000", str(seed)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    s = {k: int(v) for k, v in (t.split("=") for t in r.stdout.split())}
    assert s["tested"] > 2500 and min(s["handed_back"], s["at_h0"], s["narrow"], s["long"]) > 0
