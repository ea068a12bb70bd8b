"""Registers and scratch of the built kernels, from the code objects' own
metadata in libsejong_hip.so (no GPU needed)."""
import os
import re
import struct

import msgpack
import pytest

from sejong_amd import _native as N

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def notes(elf):
    """The AMDGPU metadata maps of an ELF code object."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + size * i + 4)
        offset, length = struct.unpack_from("<QQ", elf, shoff + size * i + 24)
        end = offset + length
        while kind == 7 and offset + 12 <= end:  # SHT_NOTE
            name, desc, tag = struct.unpack_from("<III", elf, offset)
            offset += 12 + (name + 3) // 4 * 4
            if tag == 32:  # NT_AMDGPU_METADATA
                yield msgpack.unpackb(elf[offset:offset + desc], strict_map_key=False)
            offset += (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(N.LIB_PATH):
        pytest.skip("the library is not built")
    blob = open(N.LIB_PATH, "rb").read()
    found = {}
    for at in (m.start() for m in re.finditer(re.escape(MAGIC), blob)):
        entries, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(entries):
            offset, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in triple:
                for meta in notes(blob[at + offset:at + offset + size]):
                    found.update((k[".name"], k) for k in meta["amdhsa.kernels"])
    assert len(found) > 100
    return found


def test_no_kernel_spills_its_work(kernels):
    """Spilled registers go through memory (the basis rows of ranks 33-64 with
    all their products unrolled: 2.6 KB a lane, 1.4x the time).  The attention
    backward's 10 dwords, outside its loops, are the most allowed."""
    spilled = {n: k[".private_segment_fixed_size"] for n, k in kernels.items()
               if k[".private_segment_fixed_size"] > 64}
    assert not spilled


@pytest.mark.parametrize("bm,bn,ak,bk,vgprs", [(128, 128, 0, 0, 128), (128, 128, 1, 1, 168), (128, 64, 1, 1, 128),
                                               (64, 128, 1, 1, 128)])
def test_bf16_products_keep_their_waves(kernels, bm, bn, ak, bk, vgprs):
    """sj_gemm's large bf16 tiles run four (three at 128 x 128 A^T B) waves per
    SIMD; one fewer, from a second k-step in registers, took up to 1.25x."""
    tag = f"k_gemmILi{bm}ELi{bn}ELi{ak}ELi{bk}ELi0E"
    found = [k[".vgpr_count"] for n, k in kernels.items() if tag in n]
    assert found and max(found) <= vgprs
