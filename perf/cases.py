"""Performance cases: the alignment work that programs ask of g3sa_amd.

A case names a reference, a batch of reads and the way a program calls the
library on it:

  align     Aligner.align: host codes in, alignment arrays out
  mem       what `g3a mem` does for each batch: codes, names and qualities in
            from the host, align (as one graph per batch), format the records
            on the device, copy the text out
  noalloc   as mem, through the allocation-free entry point
  resident  the batch already in HBM: align, format, copy the text out
  pairs     the batch already in HBM: align, insert-size statistics, best pair
            of hits of every read pair

The references are those of bench.py and the tests (1 Mbp uniform, 8 Mbp with
interspersed and tandem repeats, 100 Mbp and 1 Gbp with 15% and 20% repeats),
made by the project's generator and indexed on the GPU once per machine; like
the index upload, that is what a program has done before its first batch.
"""
from __future__ import annotations

import ctypes
import os
import shutil
import subprocess
import tempfile
from pathlib import Path

import numpy as np
import torch

import g3sa_amd

_REPEATS = ["--gc-mean", "0.41", "--gc-sd", "0.05", "--families", "200", "--fam-min", "300", "--fam-max", "6000",
            "--div-min", "0.05", "--div-max", "0.15"]
REFS = {
    "1m": ["--len", "1000000", "--contigs", "1", "--seed", "1"],
    "8m": ["--len", "8000000", "--contigs", "5", "--seed", "11", "--repeat-frac", "0.15", "--tandem-frac", "0.03",
           *_REPEATS],
    "100m": ["--len", "100000000", "--contigs", "5", "--seed", "11", "--repeat-frac", "0.15", *_REPEATS],
    "1g": ["--len", "1000000008", "--contigs", "24", "--seed", "21", "--repeat-frac", "0.2", *_REPEATS],
}


def _case(name, ref, reads, call, form="batched", layout="narrow", lens=(150, 150), paired=True, hard=0.0, sam=True):
    c = dict(ref=ref, reads=reads, call=call, form=form, layout=layout, len_min=lens[0], len_max=lens[1],
             paired=paired, hard=hard, sam=sam)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one read looked up from an interactive tool: latency of the whole call
        _case("one_read_1m", "1m", 1, "align", paired=False),
        # a service that answers small requests against a genome it holds
        _case("request_200_100m", "100m", 200, "mem"),
        # the same from code that may not allocate, at its largest batch
        _case("noalloc_4096_100m", "100m", 4096, "noalloc"),
        # a small run: 10k reads on a bacterial-size reference
        _case("small_10k_1m", "1m", 10000, "mem", paired=False),
        # mixed lengths (70-250 bp) with divergent reads and random tails: long extensions, ragged batches
        _case("ragged_262k_1m", "1m", 262144, "mem", lens=(70, 250), paired=False, hard=0.05),
        # the batch size of `g3a mem` on a mid-size genome, FM-index and learned seeding
        _case("mem_250k_100m", "100m", 250000, "mem"),
        _case("learned_250k_100m", "100m", 250000, "mem", form="learned"),
        # the layout that texts of 2^32 rows and more (a human genome) take
        _case("wide_250k_100m", "100m", 250000, "mem", layout="wide"),
        # one wavefront per extension task, the reference's own mapping
        _case("plain_100k_100m", "100m", 100001, "resident", form="plain", paired=False),
        # a repeat-rich reference, short reads, the reference's own record format
        _case("repeats_60k_8m", "8m", 60001, "resident", lens=(36, 101), paired=False, sam=False),
        # genome scale: the largest resident batch, learned seeding, SAM out
        _case("genome_1000k_1g", "1g", 1000000, "resident", form="learned"),
        # genome scale: pairing statistics and pair choice after the alignment, FM-index seeding
        _case("pairs_500k_1g", "1g", 500000, "pairs"),
    ]


def draw(rng):
    ref = rng.choice(["1m", "8m", "100m", "100m", "1g"])
    call = rng.choice(["align", "mem", "mem", "noalloc", "resident", "pairs"])
    form = rng.choice(["batched", "batched", "learned", "plain"])
    layout = "wide" if form == "batched" and ref != "1g" and rng.random() < 0.25 else "narrow"
    most = {"align": 2000, "noalloc": 4096}.get(call, 100000 if form == "plain" else 400000)
    reads = int(round(most ** rng.random()))
    if call == "pairs":  # statistics need some pairs
        reads = max(reads, 1000)
    paired = call == "pairs" or rng.random() < 0.5
    if paired:
        reads += reads & 1
    if rng.random() < 0.5:
        a = b = rng.choice([50, 75, 76, 100, 101, 125, 150, 151, 250])
    else:
        a = rng.randint(36, 120)
        b = rng.randint(a, 300 if call != "noalloc" else 150)
    if call == "noalloc":  # its 256 MiB hold 4096 reads of up to about 150 bases
        a, b = min(a, 151), min(b, 151)
    return _case(None, ref, reads, call, form, layout, (a, b), paired, rng.choice([0.0, 0.0, 0.05, 0.1]),
                 rng.random() < 0.8)


# ---- references and the contexts that hold their indexes

_bases: dict = {}


def _index(ref: str) -> Path:
    """Prefix of the reference's index files, made once per machine."""
    root = Path(tempfile.gettempdir()) / f"g3sa_amd_perf_{os.getuid()}"
    home = root / ref
    if not (home / "ref.g3sa").exists():
        root.mkdir(parents=True, exist_ok=True)
        tmp = Path(tempfile.mkdtemp(dir=root))
        fa = tmp / "ref.fa"
        subprocess.run([str(g3sa_amd.GEN_PATH), "ref", "-o", str(fa), *REFS[ref]], check=True)
        g3sa_amd.build_index_dev(str(fa), str(tmp / "ref"), 4)
        fa.unlink()
        try:
            tmp.rename(home)
        except OSError:  # another process was first
            shutil.rmtree(tmp, ignore_errors=True)
    return home / "ref"


def _base(case):
    """The context that loaded the reference's index, and its packed bases.

    A program loads an index once and aligns on that context's siblings, each
    with its own stream and workspace."""
    key = (case["ref"], case["layout"], case["form"] == "learned")
    if key not in _bases:
        prefix = _index(case["ref"])
        al = g3sa_amd.Aligner(str(prefix), max_reads=64, wide_layout=case["layout"] == "wide")
        if key[2]:
            al.set_learned(True)
        pac = torch.from_numpy(np.fromfile(str(prefix) + ".pac", dtype=np.uint8)).cuda()
        n = int(Path(str(prefix) + ".ann").read_text().split(None, 1)[0])
        _bases[key] = (al, pac, n)
    return _bases[key]


# ---- reads

def _reads(case, seed, pac, n_ref):
    """Codes and offsets of a batch: reads sampled from both strands with 1%
    substitutions, 0.05% indels and a few N, 1% of them from elsewhere; pairs
    point inwards with inserts of 400 +- 50; `hard` of the reads at 8%
    divergence with a random tail of 20-40 bases."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    n, lo, hi = case["reads"], case["len_min"], case["len_max"]

    def uni(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    def ints(a, b, *shape):  # [a, b)
        return torch.randint(a, b, shape, generator=g, device="cuda")

    length = ints(lo, hi + 1, n)
    rev = uni(n) < 0.5
    span = hi + 64
    start = ints(0, n_ref - 2 * span - 1024, n)
    if case["paired"]:
        ins = torch.randn(n // 2, generator=g, device="cuda").mul_(50).add_(400).round().long().clamp_(lo, 1000)
        first = rev[0::2].clone()
        rev[1::2] = ~first
        left = start[0::2].clone()  # the leftmost base of the fragment
        for k, leftmost in ((0, ~first), (1, first)):
            ln = length[k::2]
            start[k::2] = torch.where(leftmost, left, (left + ins - ln).clamp_(min=0))
    hard = uni(n) < case["hard"]
    tail = torch.where(hard, ints(20, 41, n), torch.zeros_like(length))
    sub = torch.where(hard, 0.08, 0.01)
    foreign = uni(n) < 0.01
    out = []
    for a in range(0, n, 200000):  # bounded temporaries
        b = min(n, a + 200000)
        m = b - a
        j = torch.arange(hi, device="cuda")
        e = uni(m, hi)
        insert, delete = e < 0.00025, e > 1 - 0.00025
        step = torch.ones(m, hi, dtype=torch.int32, device="cuda") - insert.int() + delete.int()
        at = torch.cumsum(step, 1) - step + start[a:b, None]
        base = (pac[(at >> 2).clamp_(max=pac.numel() - 1)] >> (6 - 2 * (at & 3)).to(torch.uint8)) & 3
        wild = ints(0, 4, m, hi).to(torch.uint8)
        base = torch.where(uni(m, hi) < sub[a:b, None], (base + 1 + wild % 3) & 3, base)
        base = torch.where(insert | foreign[a:b, None] | (j >= (length - tail)[a:b, None]), wild, base)
        base = torch.where(uni(m, hi) < 0.0002, torch.full_like(base, 4), base)
        ln = length[a:b, None]
        back = (ln - 1 - j).clamp_(min=0)
        flipped = torch.gather(base, 1, back)
        flipped = torch.where(flipped < 4, 3 - flipped, flipped)
        base = torch.where(rev[a:b, None], flipped, base)
        out.append(base[j < ln].cpu())
    off = np.zeros(n + 1, dtype=np.int32)
    off[1:] = np.cumsum(length.cpu().numpy())
    qual = torch.randint(0, 8, (int(off[-1]),), generator=g, device="cuda").mul_(5).add_(35).to(torch.uint8)
    return torch.cat(out).numpy(), off, qual.cpu().numpy()


def _names(n):
    """Names like S00001234, concatenated, with their offsets."""
    d = np.full((n, 9), ord("S"), dtype=np.uint8)
    k = np.arange(n)
    for col in range(8, 0, -1):
        d[:, col] = ord("0") + k % 10
        k = k // 10
    return d.tobytes(), np.arange(n + 1, dtype=np.int64) * 9


def prepare(case, seed):
    base, pac, n_ref = _base(case)
    seq, off, qual = _reads(case, seed, pac, n_ref)
    n = case["reads"]
    al = base.sibling(n, int(off[-1]))
    al.set_form("plain" if case["form"] == "plain" else "batched")
    al.set_graph(case["call"] == "mem")
    s = dict(case=case, al=al, seq=seq, off=off)
    if case["call"] not in ("align", "pairs"):
        names, name_off = _names(n)
        s["text"] = (names, name_off, qual.tobytes(), off.astype(np.int64))
        s["out"] = np.zeros(n * (3 * case["len_max"] + 300) + 65536, dtype=np.uint8)
    if case["call"] in ("resident", "pairs"):
        al.upload(seq, off)
        if "text" in s:
            al.upload_text(*s["text"])
    return s


def _text(s):
    """The formatted records, copied into the program's own buffer (zero past
    their end: a batch's buffer is sized before its records are known)."""
    al = s["al"]
    n = al.format(sam=s["case"]["sam"])
    if n > len(s["out"]):
        s["out"] = np.zeros(n + n // 4, dtype=np.uint8)
    rc = al.lib.g3a_copy_text(al.ctx, ctypes.c_void_p(s["out"].ctypes.data), ctypes.c_int64(len(s["out"])))
    if rc != g3sa_amd.G3A_OK:
        raise RuntimeError(f"g3a_copy_text failed ({rc})")
    return {"bytes": n, "text": s["out"]}


def _room(a, n):
    """An array in a buffer of n elements, zero past its end."""
    r = np.zeros(max(n, len(a)), dtype=a.dtype)
    r[:len(a)] = a
    return r


def run(s):
    al, call = s["al"], s["case"]["call"]
    if call == "align":
        r = al.align(s["seq"], s["off"])
        room = 4 * r.n_reads + 64
        fields = {f: _room(getattr(r, f), room) for f in (*r.FIELDS, "mapq")}
        md = np.frombuffer("\n".join(r.md).encode(), dtype=np.uint8)
        return {"aln_off": r.aln_off, **fields, "cigar": _room(r.cigar, 8 * room), "md": _room(md, 16 * room)}
    if call == "pairs":
        al.run()
        pes = al.mem_pestat(10000)
        return {"pes": pes, "rows": al.mem_pair(pes)}
    if call in ("mem", "noalloc"):
        al.upload(s["seq"], s["off"])
        al.upload_text(*s["text"])
    if call == "noalloc":
        al.run_noalloc()
    else:
        al.run()
    return _text(s)


def work(case):
    """Bytes: the batch in (codes; names and qualities where they are used)
    and its results out, and two 16-byte Occ lines for every read base, the
    least an index search that reads each base once can touch.  Operations:
    six for each cell of the two extensions of a read around its longest seed
    (the cell sets of a third of the read on either side within the band)."""
    n, length = case["reads"], (case["len_min"] + case["len_max"]) / 2
    if case["call"] == "align":
        io = length + 130
    elif case["call"] == "pairs":
        io = length + 12
    else:
        io = 2 * length + 9 + (2 * length + 60)
    side = length / 3
    return {"bytes": n * (io + 32 * length), "flops": n * 2 * side * min(side + 100, 201) * 6}
