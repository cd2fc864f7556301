"""Which extension engine runs: 16 lanes per task for few tasks, a lane per
task for many, and the lane engine alone under its autotuner."""
from __future__ import annotations

import pytest

import g3sa_amd

pytestmark = pytest.mark.gpu


def test_autotune_times_the_lane_engine(ds_c1):
    """A batch small enough for 16 lanes a task still tunes the lane engine,
    whose settings these are; the batch after it runs on 16 lanes as before."""
    _, seq, off, _ = g3sa_amd.read_fastq(str(ds_c1.reads["c3"]), limit=2000)
    with g3sa_amd.Aligner(str(ds_c1.prefix), max_reads=len(off) - 1, max_bases=int(off[-1])) as al:
        al.upload(seq, off)
        al.run()
        assert al.ext_engines() == ("group", "group")
        print("[engines] autotune", flush=True)
        al.autotune()
        assert al.ext_engines() == ("lane", "lane")
        al.run()
        assert al.ext_engines() == ("group", "group")
