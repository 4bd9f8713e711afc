"""Scratch memory and registers of the stage kernels in the built library, from
the metadata the compiler leaves in its code objects.  A stage that spills loses
10 to 100 % of its speed: the one-element FP64 forms of the 3D stage, the
covariant and the rainy stages take no scratch, at any polydeg and flux.  The
FP32 direct form keeps within the 96 registers of five waves per SIMD, without
which a third workgroup of polydeg 6 no longer fits a CU."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "trixiatmo.jl_amd",
                   "libatmo_hip.so")


def sections(elf):
    """(name offset, type, file offset, size) of an ELF64 file, and the names"""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, count, names = struct.unpack_from("<HHH", elf, 0x3A)
    raw = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + q * size) for q in range(count)]
    return [(s[0], s[1], s[4], s[5]) for s in raw], raw[names][4]


def code_objects(lib):
    """the gfx950 code objects of the offload bundles in a host library"""
    secs, names = sections(lib)
    for name, _, at, size in secs:
        if not lib[names + name:].startswith(b".hip_fatbin\0"):
            continue
        blob, pos = lib[at:at + size], 0
        while (pos := blob.find(b"__CLANG_OFFLOAD_BUNDLE__", pos)) >= 0:
            entry, (count,) = pos + 32, struct.unpack_from("<Q", blob, pos + 24)
            for _ in range(count):
                offset, length, triple = struct.unpack_from("<QQQ", blob, entry)
                if b"gfx950" in blob[entry + 24:entry + 24 + triple] and length:
                    yield blob[pos + offset:pos + offset + length]
                entry += 24 + triple
            pos += 24


def kernels(code):
    """the kernels' metadata: the AMDGPU note (type 32) of a code object"""
    for _, kind, at, size in sections(code)[0]:
        end = at + size
        while kind == 7 and at < end:
            name, desc, note = struct.unpack_from("<III", code, at)
            at += 12 + (name + 3 & ~3)
            if note == 32:
                yield from msgpack.unpackb(code[at:at + desc])["amdhsa.kernels"]
            at += desc + 3 & ~3


@pytest.fixture(scope="module")
def metadata():
    if not os.path.exists(LIB):
        raise FileNotFoundError(f"{LIB} is missing: run __graft_entry__.build()")
    with open(LIB, "rb") as f:
        lib = f.read()
    return {k[".name"]: k for code in code_objects(lib) for k in kernels(code)}


def test_stage_kernels_take_no_scratch(metadata):
    # template arguments: nodes, volume flux, gravity term, FP64, no Kahan, one
    # element a workgroup, either geometry storage
    direct = re.compile(r"e3_stage_directILi(\d)ELi\dELi\dEdLb0ELi1E[df]EE")
    seen, scratch = set(), {}
    for name, k in metadata.items():
        m = direct.search(name)
        kind = "e3 " + m[1] if m else next((s for s in ("9swe_stageI", "11rainy_stageI")
                                            if s in name), None)
        if kind:
            seen.add(kind)
            if k[".private_segment_fixed_size"]:
                scratch[name] = k[".private_segment_fixed_size"]
    assert seen == {f"e3 {n}" for n in range(2, 9)} | {"9swe_stageI", "11rainy_stageI"}
    assert not scratch, scratch


def test_fp32_direct_form_runs_five_waves_per_simd(metadata):
    direct = re.compile(r"e3_stage_directILi(\d)ELi\dELi\dEfLb[01]ELi1EfEE")
    seen, large = set(), {}
    for name, k in metadata.items():
        if m := direct.search(name):
            seen.add(int(m[1]))
            if k[".vgpr_count"] > 96 or k[".private_segment_fixed_size"]:
                large[name] = k[".vgpr_count"], k[".private_segment_fixed_size"]
    assert seen == {2, 3, 4, 6, 7, 8}  # polydeg 4 runs the pair-record form
    assert not large, large
