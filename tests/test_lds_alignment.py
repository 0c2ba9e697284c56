"""The kernels that copy 16 bytes at a time into dynamic LDS must find it 16-byte
aligned: it starts where the static LDS ends.  Reads the sizes that the compiler
recorded for the kernels of the built library."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ddc_amd", "libddcx.so")


def _code_objects(data):
    """The device ELF images of the library's offload bundles."""
    magic, pos = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (i := data.find(magic, pos)) >= 0:
        (count,) = struct.unpack_from("<Q", data, i + len(magic))
        at = i + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            if data[at + 24:at + 24 + length].startswith(b"hip") and size:
                yield data[i + offset:i + offset + size]
            at += 24 + length
        pos = i + len(magic)


def _kernels(elf):
    """The kernel descriptions of the image's metadata note."""
    (sections,) = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        head = struct.unpack_from("<IIQQQQIIQQ", elf, sections + k * entry)
        if head[1] == 7:  # SHT_NOTE
            name, desc, kind = struct.unpack_from("<III", elf, head[4])
            if kind == 32:  # NT_AMDGPU_METADATA
                at = head[4] + 12 + (name + 3) // 4 * 4
                yield from msgpack.unpackb(elf[at:at + desc])["amdhsa.kernels"]


def test_static_lds_ends_on_16_bytes():
    with open(LIB, "rb") as f:
        kernels = [k for elf in _code_objects(f.read()) for k in _kernels(elf)]
    wide = [k for k in kernels if re.search("build_tiled_kernel|build_vjp_tiled|fused_build_eval|refine_kernel", k[".name"])]
    assert len(wide) > 100
    off = {k[".name"]: k[".group_segment_fixed_size"] for k in wide if k[".group_segment_fixed_size"] % 16}
    assert not off, (len(off), sorted(set(off.values())))
