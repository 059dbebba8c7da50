"""Registers of the G4 tile kernels, from the metadata of the built library: no shape that the momentum rule can
choose keeps its totals in scratch memory (a spilled shape took 3.7 times the time of a smaller one)."""
import re
import struct

import msgpack

from dca_amd import g4acc

NT_AMDGPU_METADATA = 32


def _code_objects(data):
    """The gfx950 ELF images of the library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n, pos = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if size and b"gfx950" in name:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 1)


def _kernels(elf):
    """Kernel descriptions of a code object's metadata note."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        pos, end = offset, offset + size
        while kind == 4 and pos < end:  # PT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (namesz + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            pos = desc + (descsz + 3) // 4 * 4


def test_tile_kernels_do_not_spill_their_totals():
    """At most 128 bytes of scratch per lane; four pairs per thread (46 to 64 sites), whose shapes have one
    momentum left to give up, stay below what their three terms of one momentum need."""
    seen = 0
    for elf in _code_objects(open(g4acc.LIB_PATH, "rb").read()):
        for k in _kernels(elf):
            m = re.match(r"_ZN5g4acc14g4_pair_kernelI[fd]Li(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E", k[".name"])
            if not m:
                continue
            seen += 1
            pairs = int(m.group(2))
            assert k[".private_segment_fixed_size"] <= (352 if pairs == 4 else 128), (k[".name"], k)
    assert seen > 100
