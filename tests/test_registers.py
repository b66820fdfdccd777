"""Registers the built kernels spill to memory (their code objects' metadata):
a spill in a split kernel's chunk loop also waits for the rows in flight, so
none is let in unseen. CPU only: reads the library that the build wrote."""
import re
import struct

import pytest

import kvexp_amd


def code_objects(data: bytes):
    """The AMD GPU ELF images of the library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        pos = at + len(magic)
        (n,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24 : pos + 24 + idlen]
            pos += 24 + idlen
            if b"amdgcn" in triple and size:
                yield data[at + off : at + off + size]
        at = data.find(magic, at + len(magic))


def kernel_metadata(elf: bytes, msgpack):
    """The kernels of the image's AMDGPU metadata note."""
    shoff, shentsize, shnum = struct.unpack_from("<Q", elf, 40)[0], *struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        pos = off
        while pos < off + size:
            namesz, descsz, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (namesz + 3) // 4 * 4
            if note == 32 and elf[pos + 12 : pos + 18] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc : desc + descsz])["amdhsa.kernels"]
            pos = desc + (descsz + 3) // 4 * 4


def spills():
    msgpack = pytest.importorskip("msgpack")
    with open(kvexp_amd.LIB_PATH, "rb") as f:
        data = f.read()
    out, seen = {}, 0
    for elf in code_objects(data):
        for k in kernel_metadata(elf, msgpack):
            seen += 1
            if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]:
                out[k[".name"]] = (k[".vgpr_spill_count"], k[".private_segment_fixed_size"])
    assert seen > 300  # every instantiation of the split kernels was looked at
    return out


def test_split_kernels_spill_nothing():
    bad = {}
    for name, (regs, scratch) in spills().items():
        m = re.search(r"attn_(?:team|wave)_kernelILi(\d+)ELi(\d+)ELb(\d)ELi(\d)E", name)
        if m and regs:
            bad[m.group(0)] = (regs, scratch)
    assert not bad


def test_other_kernels_spill_only_where_named():
    """Two registers in the one-pass encoder at four chunk rows per thread."""
    bad = {n: v for n, v in spills().items()
           if not re.search(r"attn_(team|wave)_kernel", n) and not ("encode_fused_kernelILi4ELi256E" in n and v[0] <= 2)}
    assert not bad
