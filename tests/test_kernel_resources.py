"""Registers of the built kernels, from the code objects' own metadata (CPU: nothing is launched).

A work-group of decode_main is 8 waves at head_dim 64, so two of them share a CU only with at most 128 VGPRs
per lane (512 per SIMD, 4 waves).
"""

from __future__ import annotations

import os
import re
import struct
import subprocess
import sys

import msgpack
import pytest

from conftest import ROOT, load_pkg


def kernels_of(elf: bytes):
    """The kernels of one AMDGPU code object (the NT_AMDGPU_METADATA note, a msgpack map)."""
    shoff, shentsize, shnum = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, off, size = struct.unpack_from("<4xI16xQQ", elf, shoff + i * shentsize)
        if kind != 7:   # SHT_NOTE
            continue
        namesz, descsz, note = struct.unpack_from("<III", elf, off)
        if note == 32 and elf[off + 12:off + 12 + namesz].rstrip(b"\0") == b"AMDGPU":
            at = off + 12 + (namesz + 3) // 4 * 4
            return msgpack.unpackb(elf[at:at + descsz])["amdhsa.kernels"]
    return []


@pytest.fixture(scope="module")
def kernels():
    path = load_pkg().library_path()
    if not os.path.exists(path):
        subprocess.run([sys.executable, os.path.join(ROOT, "simple-inference-autoresearch_amd", "csrc", "build.py")],
                       check=True)
    lib = open(path, "rb").read()
    found = {}
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", lib):
        at = m.start()
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", lib, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", lib, pos)
            triple = lib[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in triple:
                found.update({k[".name"]: k for k in kernels_of(lib[at + off:at + off + size])})
    assert found
    return found


def pick(kernels, pattern):
    got = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert got, pattern
    return got


# decode_main<64, K/V type, q type, scale type, 8 waves, scale vectors>: 16-bit K/V, and the int8 form that
# KVCache decodes with (contiguous fp16 scales)
@pytest.mark.parametrize("pattern", [r"decode_mainILi64ENS_3F16E", r"decode_mainILi64ENS_4BF16E",
                                     r"decode_mainILi64ENS_2I8ENS_3F16ES2_Li8ELb1E",
                                     r"decode_mainILi64ENS_2I8ENS_4BF16ENS_3F16ELi8ELb1E"])
def test_head_dim_64_decode_fits_two_groups_per_cu(kernels, pattern):
    for name, k in pick(kernels, pattern).items():
        assert k[".vgpr_count"] <= 128, (name, k[".vgpr_count"])


@pytest.mark.parametrize("kernel", ["decode_main", "attn_f32_prefill"])
def test_no_register_spills(kernels, kernel):
    spills = {n: k[".vgpr_spill_count"] for n, k in pick(kernels, kernel + "I").items() if k[".vgpr_spill_count"]}
    assert not spills
