"""Registers of the built kernels, read from the metadata notes of the library's gfx950 code objects:
the streaming darker/lighter kernels keep everything in registers (private memory in their frame loop
costs them 3 to 6 %)."""
import os
import re
import struct

import msgpack

import chrono_photo_amd as cpa

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    at = blob.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", blob, at + len(MAGIC))[0]
        p = at + len(MAGIC) + 8
        for _ in range(n if n < 16 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


def _kernels(elf):
    """The kernels' metadata of one code object (note type 32, AMDGPU)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        p = off
        while p < off + size:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


def test_simple_kernels_use_no_private_memory():
    with open(os.path.join(cpa.LIB_DIR, "libchrono_hip.so"), "rb") as f:
        blob = f.read()
    found = {k[".name"]: k[".private_segment_fixed_size"] for e in _code_objects(blob) for k in _kernels(e)
             if "simple" in k[".name"]}
    assert len(found) >= 16, sorted(found)  # sample widths x channel counts x steps, at least
    assert not {n: b for n, b in found.items() if b}


def test_exchange_tiles_use_no_private_memory():
    """8-bit tiles that exchange their loads (X = 1, no sample block, the last flag set), plain and
    grouped: what spills there is written to HBM by every lane."""
    with open(os.path.join(cpa.LIB_DIR, "libchrono_hip.so"), "rb") as f:
        blob = f.read()
    pat = re.compile(r"outlier_u8_(group_)?kernelILi\dELi\d+ELi\d+ELi1ELi0ELb[01]ELb0ELb1EE")
    found = {k[".name"]: k[".private_segment_fixed_size"] for e in _code_objects(blob) for k in _kernels(e)
             if pat.search(k[".name"])}
    assert len(found) >= 96, len(found)  # 4 channel counts x 7 tiles x 2 threshold kinds, plain and grouped
    assert not {n: b for n, b in found.items() if b}
