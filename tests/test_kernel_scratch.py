"""Registers of the built kernels, read from the code objects' own metadata (no compute calls: this runs without a GPU)."""
import os
import re
import struct

import msgpack
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "parrotserve_amd", "libparrot_hip.so")


def _code_objects(blob):
    """The gfx950 ELF images in the library's offload bundles: magic, entry count, then (offset, size, name) entries."""
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        at = m.end()
        (entries,) = struct.unpack_from("<Q", blob, at)
        at += 8
        for _ in range(entries):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, at)
            name = blob[at + 24 : at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name and size:
                yield blob[m.start() + offset : m.start() + offset + size]


def _kernels(elf):
    """Kernel records of an ELF image's AMDGPU metadata note (a note is name length, payload length, type, name, payload)."""
    for m in re.finditer(rb"AMDGPU\x00\x00", elf):
        name_len, length, kind = struct.unpack_from("<III", elf, m.start() - 12)
        if name_len == 7 and kind == 32:
            return msgpack.unpackb(elf[m.end() : m.end() + length])["amdhsa.kernels"]
    return []


def test_the_fused_decode_kernels_keep_their_registers():
    """No form of the fused decode launch uses scratch: a reload in its tile loop waits for every row load in flight."""
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    blob = open(LIB, "rb").read()
    fused = {k[".name"]: k[".private_segment_fixed_size"] for elf in _code_objects(blob) for k in _kernels(elf)
             if "decode_fused_kernel" in k[".name"]}
    assert len(fused) == 36, "two types, three tiles, three kinds of suffix stream, two forms"
    assert {n: s for n, s in fused.items() if s} == {}
