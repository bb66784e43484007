"""What the layer's side branch asks of a CU, read from the built library's own kernel descriptions (no GPU needed)."""
import os
import struct

import msgpack
import pytest


def _code_objects(blob):
    """gfx950 ELF images of the library's offload bundles, one bundle to a source file."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(magic))
        entry = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            triple = blob[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(magic, at + 1)


def _kernels(elf):
    """The kernels' descriptions: the AMDGPU metadata note (type 32, MessagePack) among the program headers' notes."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        end = offset + size
        while kind == 4 and offset < end:
            name_len, data_len, note = struct.unpack_from("<III", elf, offset)
            name = offset + 12
            data = name + (name_len + 3) // 4 * 4
            if elf[name:name + name_len].rstrip(b"\0") == b"AMDGPU" and note == 32:
                yield from msgpack.unpackb(elf[data:data + data_len])["amdhsa.kernels"]
            offset = data + (data_len + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    from omni_moe.ops.hip import _lib, build
    if not os.path.exists(_lib.LIB_PATH):
        build.build_library()
    blob = open(_lib.LIB_PATH, "rb").read()
    return [k for elf in _code_objects(blob) for k in _kernels(elf)]


def test_selection_beside_the_large_tiles_takes_no_lds(kernels):
    """The ring of the 256 x 256 tiles takes all of a CU's LDS: a block of the other branch that has any waits for a CU of its own."""
    found = [k for k in kernels if "router_select_packed_kernel" in k[".name"]]
    assert len(found) >= 32
    for k in found:
        assert k[".group_segment_fixed_size"] == 0, k[".name"]


def test_selection_of_most_keys_leaves_room_for_three_waves(kernels):
    """More than 512 keys a half, up to 256 candidates: with a few more registers than 168 a SIMD holds two waves instead of three, which took 14 % longer."""
    found = [k for k in kernels if any(f"router_select_packed_kernelILi{dt}ELi16ELi{c}E" in k[".name"] for dt in (0, 1) for c in (1, 2, 4))]
    assert len(found) == 6
    for k in found:
        assert k[".vgpr_count"] + k.get(".agpr_count", 0) <= 168, k[".name"]
