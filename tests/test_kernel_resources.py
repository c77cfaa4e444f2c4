"""No GEMV kernel keeps registers in scratch memory.

The row tiles, waves and chunks per wave of a chunked GEMV instantiation set
its registers per lane; one past the limit of its workgroup size still
compiles, to a kernel that moves them through memory in every chunk (fused
q8_0 12288x7168 at batch 8: 151 us with 99 spilled registers, 58 without).
The built library carries each kernel's counts in its code objects' notes."""
from __future__ import annotations

import struct

import msgpack

from qwowl35_amd import build


def _kernels(blob: bytes):
    """The kernels of every code object (ELF64 with an AMDGPU metadata note) in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", blob, pos - 8)[0]):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, pos)
            pos += 24 + name_len
            elf = blob[at + offset:at + offset + size]
            if elf[:4] != b"\x7fELF":
                continue
            sections, entry, n = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
            for i in range(n):
                kind, _, _, start, length = struct.unpack_from("<IQQQQ", elf, sections + i * entry + 4)
                while kind == 7 and length >= 12:  # SHT_NOTE
                    owner, desc, note = struct.unpack_from("<III", elf, start)
                    body = start + 12 + (owner + 3) // 4 * 4
                    if note == 32:  # NT_AMDGPU_METADATA
                        yield from msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]
                    end = body + (desc + 3) // 4 * 4
                    length -= end - start
                    start = end
        at = blob.find(magic, pos)


def test_no_gemv_kernel_spills_registers():
    kernels = [k for k in _kernels(build.LIB.read_bytes()) if "_gemv" in k[".name"]]
    assert len(kernels) > 100
    spilled = {k[".name"]: k[".vgpr_spill_count"] for k in kernels if k[".vgpr_spill_count"]}
    assert not spilled, spilled
