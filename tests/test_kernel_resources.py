"""What the compiler gave each kernel of the built library, from the metadata of its own code objects."""
import struct

import pytest


def _code_objects(blob):
    """The gfx950 code objects in a host library: every offload bundle's entries, by the bundle's header."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(count if count < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            if b"gfx950" in blob[pos + 24:pos + 24 + length]:
                yield blob[at + offset:at + offset + size]
            pos += 24 + length
        at += len(magic)


def _kernels(elf, msgpack):
    """The kernels of a code object: the message-pack map in its AMDGPU metadata note."""
    sections, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, sections + i * size + 4)
        offset, length = struct.unpack_from("<QQ", elf, sections + i * size + 24)
        pos = offset
        while kind == 7 and pos < offset + length:                  # SHT_NOTE
            name, desc, what = struct.unpack_from("<III", elf, pos)
            start = pos + 12 + (name + 3) // 4 * 4
            if what == 32:                                          # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]
            pos = start + (desc + 3) // 4 * 4


def test_no_gemm_kernel_keeps_registers_in_scratch_memory():
    """A reload from scratch waits for every transfer of the tiles under way (they complete in order)."""
    msgpack = pytest.importorskip("msgpack")
    from hpfp8 import _lib
    with open(_lib.LIB_PATH, "rb") as f:
        kernels = [k for elf in _code_objects(f.read()) for k in _kernels(elf, msgpack)]
    gemm = [k for k in kernels if "gemm" in k[".name"]]
    assert len(gemm) > 50
    assert not [(k[".name"], k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for k in gemm
                if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]]
