"""Seeding by a group of lanes (g3a_seed.h) on the CPU: its lanes as fibers,
in the narrow, the wide and the full-suffix-array form, against the one-thread
seeding rounds (tests/seed_group_check.cpp)."""
from __future__ import annotations

import subprocess

import pytest

import g3sa_amd
from conftest import ROOT, gen


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    out = tmp_path_factory.mktemp("seed_group") / "seed_group_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-I", str(ROOT), "-o", str(out),
                    str(ROOT / "tests" / "seed_group_check.cpp"), str(ROOT / "g3sa_amd" / "csrc" / "index_io.cpp")],
                   check=True, capture_output=True)
    return out


@pytest.fixture(scope="module")
def repeats(built, tmp_path_factory):
    d = tmp_path_factory.mktemp("seed_group_ref")
    gen("ref", "-o", str(d / "r.fa"), "--len", "600000", "--contigs", "3", "--seed", "5", "--repeat-frac", "0.2",
        "--families", "50", "--fam-min", "300", "--fam-max", "6000", "--div-min", "0.0", "--div-max", "0.05",
        "--tandem-frac", "0.03")
    g3sa_amd.build_index(str(d / "r.fa"), str(d / "r"), 16)
    return d / "r"


@pytest.mark.parametrize("min_seed_len", [9, 12, 13, 19, 31])
def test_seed_group_equals_one_thread(checker, repeats, min_seed_len):
    """Around the k-mer table's 12 bases (at most 12: no table in the backward
    phases), the default and a long one; reads of 0 to 320 bases."""
    r = subprocess.run([str(checker), str(repeats), "300", str(min_seed_len)], capture_output=True, text=True,
                       timeout=600)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
    s = {k: float(v) for k, v in (t.split("=") for t in r.stdout.split()[1:])}
    # With seeds longer than the table's 12 bases a 16-lane group gives up the
    # reads of one repeated word (one in 29) and some of the text's tandem
    # repeats (3% of it): a tenth at most.  Shorter seeds are many more and may
    # fill the 64 output slots of a long read, but not of the shorter half.
    # A third of the 233 text reads of 36 bases or more have no errors, so each
    # of those that is not given up has an interval.
    most = 30 if min_seed_len > 12 else 150
    for form in ("narrow", "wide", "text"):
        assert s[f"given_up_{form}"] <= most, form
        assert s[f"compared_{form}"] >= 300 * 6 // 7 * 10 // 11 // 3 - 30, form
