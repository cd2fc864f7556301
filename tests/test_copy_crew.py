"""The copying threads of the host transfers (g3a_copy.h): chunk and piece
remainders, slot reuse with transfers awaited as late as allowed, and errors
part way (tests/copy_crew_check.cpp)."""
from __future__ import annotations

import subprocess

from conftest import ROOT


def test_copy_crew(tmp_path):
    exe = tmp_path / "copy_crew_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", str(ROOT), "-o", str(exe),
                    str(ROOT / "tests" / "copy_crew_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
