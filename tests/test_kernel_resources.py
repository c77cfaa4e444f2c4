"""No GEMV kernel keeps registers in scratch memory.

The row tiles, waves and chunks per wave of a chunked GEMV instantiation set
its registers per lane; one past the limit of its workgroup size still
compiles, to a kernel that moves them through memory in every chunk (fused
q8_0 12288x7168 at batch 8: 151 us with 99 spilled registers, 58 without).
The built library carries each kernel's counts in its code objects' notes."""
from __future__ import annotations

import re
import struct

import msgpack

from qwowl35_amd import build
from tests.test_plan_coverage import GF2, Q4K, Q5K, Q6K, Q8, kernel


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


def test_every_chunked_gemv_kernel_is_launched():
    """No instantiation of the chunked kernel that no shape launches (GF4 left
    out: its plain ones are the greedy head's, which is not described here)."""
    built = set()
    for k in _kernels(build.LIB.read_bytes()):
        m = re.search(r"(kq_mfma_gemv(?:_long)?)I(\w+?)EEv", k[".name"])
        if m:
            args = [n or ("true" if b == "1" else "false") for n, b in re.findall(r"Li(\d+)E|Lb(\d)", m.group(2))]
            if args[0] != "2" and args[-1] == "false":  # (the other half takes an AWQ multiplier)
                built.add(f"{m.group(1)}<{', '.join(args)}>")
    tiles = [1, 257, 385, 513, 640, 769, 832, 1025, 1089, 1281, 1344, 1537, 1664, 2049, 3073, 4096, 4097, 6250]
    chunks = [2, 4, 6, 8, 10, 12, 14, 16, 18, 24, 26, 28, 32, 40, 48, 50, 52, 68]
    launched = set()
    for t in (GF2, Q8, Q4K, Q5K, Q6K):
        for swiglu in (False, True):
            for n in tiles if not (swiglu and t == Q6K) else []:
                for c in chunks:
                    for nb in (1, 2, 3, 8):
                        launched.add(kernel(t, 16 * n, 256 * c, nb, swiglu=swiglu))
                        if c >= 48:
                            launched.add(kernel(t, 16 * n, 256 * c, nb, swiglu=swiglu, ws=True).split("+")[0])
    assert built and built <= launched, sorted(built - launched)
