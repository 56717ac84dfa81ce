"""Registers of the built kernels, from the metadata of the library's own code
objects: what the decode kernels' occupancy rests on (512 vector registers a
SIMD lane are shared by its waves in units of eight)."""
from __future__ import annotations

import re
import struct

import pytest

from unifur_amd import _lib

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    for m in re.finditer(MAGIC, blob):
        base = m.start()
        count, at = struct.unpack_from("<Q", blob, base + len(MAGIC))[0], base + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, at)
            name = blob[at + 24:at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name and size:
                yield blob[base + offset:base + offset + size]


def metadata(elf):
    """The kernels' metadata (a msgpack note) of one code object."""
    msgpack = pytest.importorskip("msgpack")
    phoff, phentsize, phnum = (struct.unpack_from(f, elf, o)[0] for f, o in (("<Q", 32), ("<H", 54), ("<H", 56)))
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        at, end = offset, offset + size
        while kind == 4 and at + 12 <= end:  # PT_NOTE
            name_size, desc_size, note = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (name_size + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                return msgpack.unpackb(elf[desc:desc + desc_size])["amdhsa.kernels"]
            at = desc + (desc_size + 3) // 4 * 4
    return []


@pytest.fixture(scope="module")
def kernels():
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for elf in code_objects(blob) for k in metadata(elf)}
    assert found, "no gfx950 kernel metadata in the library"
    return found


def matching(kernels, pattern):
    found = [k for name, k in kernels.items() if re.search(pattern, name)]
    assert found, pattern
    return found


# skinny_kernel<NT, W, D, S, DQ, PAIR, XF32, NORM>
def test_f32_pair_of_one_token_tile_runs_three_waves(kernels):
    for k in matching(kernels, r"skinny_kernelILi1ELi[48]ELi2ELi4ELb1ELb1ELb1ELb1E"):
        assert k[".vgpr_count"] <= 168 and k[".vgpr_spill_count"] == 0, k[".name"]


def test_bf16_pair_of_four_token_tiles_spills_no_more(kernels):
    for k in matching(kernels, r"skinny_kernelILi4ELi8ELi2ELi2ELb1ELb1ELb0ELb1E"):
        assert k[".vgpr_spill_count"] <= 4, k[".name"]


def test_f32_gemm_runs_two_waves_without_spills(kernels):
    # gemm_f32_kernel<RT, DQ, STRIPED, TRANS, XBF, SERIAL>; with SERIAL a grid has at most a workgroup a CU
    for k in matching(kernels, r"gemm_f32_kernelILi[24]E(Lb[01]E){4}Lb0E"):
        assert k[".vgpr_count"] <= 256 and k[".vgpr_spill_count"] == 0, k[".name"]
    for k in matching(kernels, r"gemm_f32_kernelILi[24]E(Lb[01]E){4}Lb1E"):
        assert k[".vgpr_count"] <= 512 and k[".vgpr_spill_count"] == 0, k[".name"]
