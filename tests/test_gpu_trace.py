"""Traceback of gapped alignments at the widths of the group kernels: reads
with an insertion or deletion of 1 to 70 bases (bands of up to 16, 32, 64 and
128 columns and wider) at lengths up to the limit, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _batch, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [70, 151, 319, 320])
def test_gapped_alignments(ds_c1, oracle, length):
    text = "".join(ln.strip() for ln in open(ds_c1.fasta) if not ln.startswith(">")).upper()
    ref = np.array(["ACGTN".index(c) for c in text], dtype=np.uint8)
    rng = np.random.default_rng(length)
    reads = []
    for gap in [1, 2, 3, 4, 5, 8, 11, 12, 13, 20, 27, 28, 29, 40, 59, 60, 61, 70]:
        for place in (3, 2):
            p = int(rng.integers(1000, len(ref) - 1000))
            at = length // place
            r = np.concatenate([ref[p:p + at], ref[p + at + gap:p + gap + length]])  # deletion
            reads.append(r.copy())
            ins = rng.integers(0, 4, gap).astype(np.uint8)
            r = np.concatenate([ref[p:p + at], ins, ref[p + at:p + length]])[:length]  # insertion
            r[rng.integers(0, length, 2)] = rng.integers(0, 5, 2)
            reads.append(r)
            reads.append((3 - reads[-2][::-1]).astype(np.uint8))  # the other strand
    seq, off = _batch(reads)
    print(f"[trace] {len(reads)} reads of {length}", flush=True)
    run_both(ds_c1, oracle, seq, off, f"gapped, {length} bases")
