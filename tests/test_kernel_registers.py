"""The kernels whose waits count their own copies in flight must keep every vector register: a reload of a spilled one waits for all
of those copies, and a register that an assembly statement fills asynchronously would be spilled before its value has arrived."""
import os
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-kunlun_amd", "lib", "libkmoe.so")


def _code_objects(blob):
    """The gfx950 ELF images among the offload bundles of a library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        count, pos = struct.unpack_from("<Q", blob, at + len(magic))[0], at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<3Q", blob, pos)
            if b"gfx950" in blob[pos + 24:pos + 24 + length]:
                yield blob[at + offset:at + offset + size]
            pos += 24 + length
        at += len(magic)


def _kernels(elf):
    """The kernel entries of an image's metadata note."""
    table, (size, count) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<2H", elf, 58)
    for i in range(count):
        kind, _, _, start, length = struct.unpack_from("<I4Q", elf, table + i * size + 4)
        end = start + length
        while kind == 7 and start < end:  # notes
            name, desc, what = struct.unpack_from("<3I", elf, start)
            body = start + 12 + (name + 3) // 4 * 4
            if what == 32 and elf[start + 12:start + 18] == b"AMDGPU":
                yield from msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]
            start = body + (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    return [k for elf in _code_objects(open(LIB, "rb").read()) for k in _kernels(elf)]


def test_macro_tiles_spill_nothing(kernels):
    tiles = [k for k in kernels if "macro_tile_kernel" in k[".name"]]
    assert len(tiles) == 16
    assert not {k[".name"]: k[".vgpr_spill_count"] for k in tiles if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
