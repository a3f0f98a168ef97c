"""What the built kernels ask of a launch, read from their descriptors.

A kernel that is given the dispatch packet reads it from host memory, every
workgroup for itself.  No kernel here needs it; the compiler asks for it when it
keeps a private array in LDS.
"""

from __future__ import annotations

import os
import struct

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "nanochat-filter_amd", "nanochat_amd", "libnanochat_filter_amd.so")
_BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
_DISPATCH_PTR = 1 << 1  # kernel_code_properties: ENABLE_SGPR_DISPATCH_PTR


def _sections(elf: bytes):
    """(name, type, file offset, size, link, entry size) of an ELF64 file's sections."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    size, n, strndx = struct.unpack_from("<HHH", elf, 58)
    raw = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * size) for i in range(n)]
    names = raw[strndx][4]

    def name(off):
        return elf[names + off:elf.index(b"\0", names + off)].decode()

    return [(name(r[0]), r[1], r[3], r[4], r[5], r[6], r[9]) for r in raw]


def _code_objects(lib: bytes):
    fat = next(s for s in _sections(lib) if s[0] == ".hip_fatbin")
    blob = lib[fat[3]:fat[3] + fat[4]]
    at = blob.find(_BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(_BUNDLE))
        pos = at + len(_BUNDLE) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(_BUNDLE, at + 1)


def _kernel_properties(elf: bytes):
    """(kernel, kernel_code_properties) of one code object."""
    secs = _sections(elf)
    for _, kind, _, off, size, link, ent in secs:
        if kind != 11:  # SHT_DYNSYM
            continue
        strs = secs[link][3]
        for i in range(size // ent):
            nm, _, _, shndx, value, _ = struct.unpack_from("<IBBHQQ", elf, off + i * ent)
            name = elf[strs + nm:elf.index(b"\0", strs + nm)].decode()
            if name.endswith(".kd"):
                _, _, addr, base, _, _, _ = secs[shndx]
                yield name[:-3], struct.unpack_from("<H", elf, base + (value - addr) + 56)[0]


def test_no_kernel_reads_the_dispatch_packet():
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    with open(LIB, "rb") as f:
        lib = f.read()
    props = [p for co in _code_objects(lib) for p in _kernel_properties(co)]
    assert len(props) > 100
    assert [k for k, p in props if p & _DISPATCH_PTR] == []
