"""The seeding kernels' intervals against the oracle's seeding rounds, at the
read lengths and seed lengths where the group search can go wrong."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import g3sa_amd
from test_gpu_learned import _intervals_equal
from test_gpu_parity import _batch

pytestmark = pytest.mark.gpu


def _reads(ds):
    """Lengths 0 to 40 and the limit's neighbours, matches with and without
    substitutions and N, and repeats of one to three bases."""
    _, seq, off, _ = g3sa_amd.read_fastq(str(ds.reads["main"]), limit=400)
    rng = np.random.default_rng(3)
    pool = [seq[off[i]:off[i + 1]] for i in range(len(off) - 1)]
    reads = [pool[n][:n] for n in range(41)] + [pool[50 + n][:63 + n] for n in range(4)]
    for n in (317, 318, 319, 320):
        reads.append(np.concatenate([pool[n - 200], pool[n - 190], pool[n - 180]])[:n])
    for t in (1, 2, 3):
        reads += [(np.arange(n) % t).astype(np.uint8) for n in (12, 19, 20, 150, 320)]
    for i in range(100, 300):
        r = pool[i].copy()
        r[rng.integers(0, len(r), i % 4)] = 4
        reads.append(r)
    return reads + pool[300:]


@pytest.mark.parametrize("form", ["narrow", "wide", "learned"])
@pytest.mark.parametrize("min_seed_len", [11, 12, 13, 19])
def test_seeding_edges(ds_rep, oracle, form, min_seed_len):
    seq, off = _batch(_reads(ds_rep))
    n = len(off) - 1
    oo = type(oracle.opt)()
    C.pointer(oo)[0] = oracle.opt
    oo.min_seed_len = min_seed_len
    go = g3sa_amd.default_opt()
    go.min_seed_len = min_seed_len
    idx = oracle.load(ds_rep.prefix)
    keep, oracle.opt = oracle.opt, oo
    try:
        ref = [oracle.seed_intervals(idx, seq[off[i]:off[i + 1]]) for i in range(n)]
    finally:
        oracle.opt = keep
        oracle.lib.orc_index_free(idx)
    counts = np.array([len(r) for r in ref], dtype=np.int32)
    flat = np.array([(k, s, m, e) for r in ref for (k, _l, s, m, e) in r], dtype=np.int64).reshape(-1, 4)
    with g3sa_amd.Aligner(str(ds_rep.prefix), max_reads=n, max_bases=int(off[-1]), opt=go,
                          wide_layout=form == "wide") as al:
        if form == "learned":
            al.set_learned(1)
        print(f"[seed] {form}, min_seed_len {min_seed_len}: {n} reads", flush=True)
        al.align(seq, off)
        _intervals_equal((counts, flat), al.intervals(), f"{form} min_seed_len {min_seed_len}")


@pytest.mark.parametrize("form", ["narrow", "wide", "learned"])
def test_ordinary_reads_stay_on_16_lanes(ds_c1, form):
    """A group that gives up leaves its read to the slow path, whose output is
    the same: reads of 150 bases at 1% substitutions on a text without repeats
    have short lists and few matches, so hardly any may go there."""
    _, seq, off, _ = g3sa_amd.read_fastq(str(ds_c1.reads["main"]))
    n = len(off) - 1
    with g3sa_amd.Aligner(str(ds_c1.prefix), max_reads=n, max_bases=int(off[-1]), wide_layout=form == "wide") as al:
        if form == "learned":
            al.set_learned(1)
        got = al.align(seq, off)
    assert got.work["n_slow_reads"] <= n // 100
