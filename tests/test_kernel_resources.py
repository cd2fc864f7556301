"""Registers of the built kernels, from the code objects' own metadata.

A grid of four wavefronts a SIMD needs kernels of at most 128 of its 512
registers a lane; one register more and every grid runs with three.
"""
from __future__ import annotations

import struct

import msgpack
import pytest


def _kernels(lib) -> dict:
    """Metadata of every kernel of the library's gfx950 code objects, by name."""
    data, out, at = lib.read_bytes(), {}, 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        p = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, p - 8)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if data[p + 24:p + 24 + n].endswith(b"gfx950"):
                out.update(_elf_kernels(data[at + off:at + off + size]))
            p += 24 + n
        at += len(magic)
    return out


def _elf_kernels(elf: bytes) -> dict:
    sh, (esz, n) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
    for k in range(n):
        kind, off, size = (struct.unpack_from("<I", elf, sh + k * esz + 4)[0],
                           *struct.unpack_from("<QQ", elf, sh + k * esz + 24))
        while kind == 7 and size > 0:  # SHT_NOTE
            ns, ds, t = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (ns + 3 & ~3)
            if t == 32:  # NT_AMDGPU_METADATA
                meta = msgpack.unpackb(elf[desc:desc + ds], raw=False)
                return {m[".name"]: m for m in meta["amdhsa.kernels"]}
            step = desc + (ds + 3 & ~3) - off
            off, size = off + step, size - step
    return {}


@pytest.mark.parametrize("sym", [0, 1])
@pytest.mark.parametrize("packed", [0, 1])
def test_lane_engine_leaves_four_wavefronts_a_simd(built, sym, packed):
    k = _kernels(built / "libg3a.so")[f"_ZN3g3a10k_ext_laneILi16ELb{sym}ELb{packed}EEEvNS_11ExtSideArgsE"]
    assert k[".vgpr_count"] <= 128
    assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0
