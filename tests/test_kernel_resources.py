"""Registers of the built operator kernels, from the metadata that the compiler
leaves in the library's code objects."""
import re
import struct
from pathlib import Path

import msgpack
import pytest

LIB = Path(__file__).resolve().parents[1] / "nekbench_amd" / "libnbx.so"


def code_objects(data):
    """The gfx950 ELF images of every offload bundle in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + 1)


def kernels(elf):
    """The kernel descriptions of one ELF image (its AMDGPU metadata note)."""
    phoff, phsize, phnum = struct.unpack_from("<Q", elf, 32)[0], *struct.unpack_from("<HH", elf, 54)
    for k in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + k * phsize)
        if kind != 4:  # PT_NOTE
            continue
        p, end = offset, offset + size
        while p + 12 <= end:
            nlen, dlen, tag = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if tag == 32:  # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[d:d + dlen])["amdhsa.kernels"]
            p = d + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def built(nbx):
    out = {}
    for elf in code_objects(LIB.read_bytes()):
        for k in kernels(elf):
            out[k[".name"]] = k
    return out


def test_operator_rows_of_D_do_not_spill(built):
    """The rows of D are scalar operands that are read row by row: no form of
    the one-field operator spills them (the FP64 Helmholtz form at N = 15, with
    64 scalars of two rows, may spill a few addresses)."""
    seen = 0
    for name, k in built.items():
        m = re.match(r"_ZN3nbx8k_axhelmI([df])Li(\d+)ELi1ELb([01])E", name)
        if m:
            seen += 1
            allowed = 32 if m[1] == "d" and m[2] == "16" else 0
            assert k[".sgpr_spill_count"] <= allowed, (name, k[".sgpr_spill_count"])
            assert k[".vgpr_spill_count"] == 0, (name, k[".vgpr_spill_count"])
    assert seen == 15 * 2 * (2 + 2 + 1)  # orders, forms; whole and list in FP64 and FP32, whole with bf16 geometry


def test_forms_that_no_call_reaches_are_not_built(built):
    """FP32 geometry with bf16 operands has no precision of its own, and the
    three-field PCG form takes a thread group per field at every mesh size for
    these orders."""
    mma = [n for n in built if "14k_axhelm_mma16I" in n]
    assert mma and not [n for n in mma if "EfNS_6OpBf16E" in n]
    turn = {m.groups() for m in (re.match(r"_ZN3nbx12k_axhelm_pcgILi(\d+)ELi3ELb([01])E([df])(\w)Li0E", n) for n in built)
            if m}
    assert ("8", "1", "d", "d") in turn and ("15", "1", "d", "d") in turn
    assert not [t for t in turn if t[2] == "d" and t[0] in ("12", "13", "14")]
    assert not [t for t in turn if t[3] == "f" and int(t[0]) >= 9]
