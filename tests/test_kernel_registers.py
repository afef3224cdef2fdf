"""What the compiler gave the kernels that are built around a number of workgroups per compute unit, from the metadata of the
built library, without a GPU."""

import os
import re
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor-product-attention-jax_amd", "lib", "libtpa_gfx950.so")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(BUNDLE)
    while at >= 0:
        (count,), place = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, place)
            if b"gfx950" in blob[place + 24 : place + 24 + length]:
                yield blob[at + offset : at + offset + size]
            place += 24 + length
        at = blob.find(BUNDLE, at + 24)


@pytest.fixture(scope="module")
def kernels():
    """name -> its metadata (NT_AMDGPU_METADATA notes of the ELF code objects)"""
    found = {}
    for obj in _code_objects(open(LIB, "rb").read()):
        (table,), (entry, count) = struct.unpack_from("<Q", obj, 0x28), struct.unpack_from("<HH", obj, 0x3A)
        for i in range(count):
            (kind,), (offset, size) = struct.unpack_from("<I", obj, table + i * entry + 4), struct.unpack_from("<QQ", obj, table + i * entry + 0x18)
            at = offset
            while kind == 7 and at < offset + size:
                name, desc, note = struct.unpack_from("<III", obj, at)
                body = at + 12 + (name + 3) // 4 * 4
                if note == 32:
                    found.update((k[".name"], k) for k in msgpack.unpackb(obj[body : body + desc])["amdhsa.kernels"])
                at = body + (desc + 3) // 4 * 4
    assert found
    return found


def test_decode_with_rows_side_by_side_keeps_two_workgroups_at_head_size_64(kernels):
    """256 registers (both kinds together) are two waves per SIMD: two workgroups of four waves on a compute unit."""
    name = re.compile(r"13decode_kernelILi64ELi(\d+)ELb[01]ELi1ELNS0_5ReadsE\dELb1EE")
    side = {n: k for n, k in kernels.items() if name.search(n)}
    assert {int(name.search(n).group(1)) for n in side} == {1, 2, 4, 8, 16, 32}
    assert {n: k[".vgpr_count"] for n, k in side.items() if k[".vgpr_count"] > 256} == {}
    assert all(k[".private_segment_fixed_size"] == 0 for k in side.values()), "scratch memory"
