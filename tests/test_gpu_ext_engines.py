"""Which extension engine runs: 16 lanes per task for few tasks, a lane per
task for many, and the lane engine alone under its autotuner."""
from __future__ import annotations

import numpy as np
import pytest

import g3sa_amd
from test_gpu_parity import _with_scoring

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


def test_plain_form_fills_the_chip_outside_the_16_bit_domain(ds_c1, oracle):
    """At a mismatch score of -9 every task takes the one-wavefront kernel.  The
    plain form gives each a block; the batched form's 8 blocks a compute unit
    leave three quarters of the wavefronts' places empty and take 2.3 times as
    long on a full chip."""
    _, seq, off, _ = g3sa_amd.read_fastq(str(ds_c1.reads["main"]))
    seq, n = np.tile(seq[:off[-1]], 8), 8 * (len(off) - 1)
    off = np.concatenate([off[:-1] + k * off[-1] for k in range(8)] + [[8 * off[-1]]]).astype(np.int32)
    ms = {}
    with g3sa_amd.Aligner(str(ds_c1.prefix), max_reads=n, max_bases=int(off[-1]), opt=_with_scoring(oracle, b=9)[1]) as al:
        al.set_tuning(16, 8, 8)
        al.upload(seq, off)
        for form in ("plain", "batched"):
            al.set_form(form)
            print(f"[engines] {form}, {n} reads", flush=True)
            for _ in range(3):
                al.run()
            assert al.ext_engines() == (None, None)
            ms[form] = al.stats()["ms"]["extend"]
    assert ms["plain"] < 0.7 * ms["batched"], ms
