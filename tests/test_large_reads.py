"""Chaining and region filter of one read by a wavefront (g3a_chain.h,
g3a_region.h) on the CPU: their lanes as fibers, against the one-thread code,
on random seed lists and regions (tests/chain_group_check.cpp,
tests/region_group_check.cpp)."""
from __future__ import annotations

import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("check,reads,seed", [("chain_group_check", 10, 1), ("chain_group_check", 10, 2),
                                              ("region_group_check", 60, 1), ("region_group_check", 60, 2)])
def test_wavefront_equals_one_thread(tmp_path, check, reads, seed):
    exe = tmp_path / check
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(ROOT), "-o", str(exe),
                    str(ROOT / "tests" / f"{check}.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe), str(reads), str(seed)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
    s = {k: int(v) for k, v in (t.split("=") for t in r.stdout.split()[1:])}
    assert min(s.values()) > 0
