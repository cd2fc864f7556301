"""Global alignment by a group of lanes (g3a_trace.h) on the CPU: its lanes
as fibers, against the one-thread alignment (tests/trace_group_check.cpp), in
all four widths, with three scorings, N, long indels and short reads."""
from __future__ import annotations

import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_trace_group_equals_one_thread(tmp_path, seed):
    exe = tmp_path / "trace_group_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(ROOT), "-o", str(exe),
                    str(ROOT / "tests" / "trace_group_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe), "400", str(seed)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
    s = {k: int(v) for k, v in (t.split("=") for t in r.stdout.split()[1:])}
    assert min(s["by16"], s["by32"], s["by64"], s["by128"], s["gapped"]) > 0
