"""The matrix-core GEMM's forms are chosen so that their accumulators and operands fit the registers: none keeps any of them in scratch
memory (read from the metadata of the built library; no GPU needed)."""
import os
import re
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "densecore_amd", "libmi355q4k.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    for at in (m.start() for m in re.finditer(MAGIC, blob)):
        count, = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(count):
            offset, size, idlen = struct.unpack_from("<3Q", blob, pos)
            if blob[pos + 24:pos + 24 + idlen].startswith(b"hip") and size:
                yield blob[at + offset:at + offset + size]
            pos += 24 + idlen


def kernels(elf):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<2H", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        at, = struct.unpack_from("<Q", elf, shoff + i * shentsize + 0x18)
        namesz, descsz, note = struct.unpack_from("<3I", elf, at)
        if note == 32:  # NT_AMDGPU_METADATA
            desc = at + 12 + (namesz + 3) // 4 * 4
            yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]


@pytest.mark.skipif(not os.path.exists(LIB), reason="the library is not built")
def test_no_gemm_form_spills():
    gemms = [k for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf) if "gemm" in k[".name"]]
    assert len(gemms) > 60
    assert not [(k[".name"], k[".vgpr_spill_count"]) for k in gemms if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]
