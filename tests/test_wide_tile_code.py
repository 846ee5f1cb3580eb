"""The wide tiles of the direct form issue their matrix instructions from inline assembly, which the compiler does not know as such: it
waits for none of their results.  What the source cannot promise is looked up in the built code: between the first and the last of
them nothing else touches an accumulator, a wait is between the last and the first read, and no operand is written right before its use."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from pytorch_winoconv_amd import _lib

OBJDUMP = shutil.which("llvm-objdump", path=os.environ.get("ROCM_PATH", "/opt/rocm") + "/llvm/bin") or shutil.which("llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The GPU code objects of a shared library: bundles of (offset, size, target) entries"""
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + n]:
                yield data[at + offset:at + offset + size]
            entry += 24 + n
        at = data.find(MAGIC, at + len(MAGIC))


def _registers(text, kind):
    """The numbers of the registers of `kind` ('a' or 'v') named in operands such as v7, a[0:3]"""
    found = set()
    for one, first, last in re.findall(r"\b%s(?:(\d+)\b|\[(\d+):(\d+)\])" % kind, text):
        found.update([int(one)] if one else range(int(first), int(last) + 1))
    return found


def _unguarded(lines):
    """What stands in the way of the matrix instructions among `lines` of assembly"""
    wrong = [l for l in lines if l.startswith("scratch_")]
    mfma = [i for i, l in enumerate(lines) if l.startswith("v_mfma")]
    for i, l in enumerate(lines[mfma[0]:mfma[-1]], mfma[0]):
        if i not in mfma and _registers(l, "a"):
            wrong.append(l)
    for i in mfma:
        read = _registers(lines[i].split(",", 1)[1], "v")
        wrong += [l for l in lines[max(i - 3, 0):i] if l.startswith("v_") and not l.startswith("v_mfma") and _registers(l.split(",")[0], "v") & read]
    waited = False
    for l in lines[mfma[-1] + 1:]:
        waited = waited or l == "s_nop 15"
        if _registers(l, "a"):
            return wrong + ([] if waited else [l])
    return wrong + ["no accumulator is read"]


def test_what_counts_as_unguarded():
    good = ["v_accvgpr_write_b32 a0, 0", "ds_read_b128 v[0:3], v9", "v_mfma_f32_16x16x32_f16 a[0:3], v[0:3], v[4:7], a[0:3]", "v_add_u32_e32 v9, 1, v9", "s_nop 0",
            "v_mfma_f32_16x16x32_f16 a[4:7], v[0:3], v[4:7], a[4:7]", "s_nop 15", "v_accvgpr_read_b32 v0, a0"]
    assert _unguarded(good) == []
    assert _unguarded(good[:3] + ["v_accvgpr_read_b32 v10, a3"] + good[3:])
    assert _unguarded(good[:2] + ["v_mov_b32_e32 v6, v20"] + good[2:])
    assert _unguarded(good[:6] + good[7:])
    assert _unguarded(good[:4] + ["scratch_store_dword off, v9, s32"] + good[4:])


def test_nothing_touches_the_accumulators_of_the_wide_tiles(tmp_path):
    if OBJDUMP is None:
        pytest.skip("no llvm-objdump")
    with open(_lib.LIB_PATH, "rb") as f:
        objects = [o for o in _code_objects(f.read()) if b"direct_wide_kernel" in o]
    assert len(objects) == 1
    path = tmp_path / "code.o"
    path.write_bytes(objects[0])
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True, capture_output=True, text=True).stdout
    kernels = 0
    for name, body in re.findall(r"^<?([^\n]*direct_wide_kernel[^\n>]*)>?:\n(.*?)(?=^<|^\S[^\n]*:\n|\Z)", text, re.S | re.M):
        lines = [l.split("//")[0].strip() for l in body.split("\n")]
        assert _unguarded([l for l in lines if l]) == [], name
        kernels += 1
    assert kernels == 6          # three widths, two types
