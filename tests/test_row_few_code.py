"""The row form's kernel for few tiles (conv_row_few.hip) without a GPU: it keeps what it works on in registers, looked up in the built code, and the
filters that it takes as they are."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest
import torch

from pytorch_winoconv_amd import _lib, engine
from test_wide_tile_code import _code_objects

READELF = shutil.which("llvm-readelf", path=os.environ.get("ROCM_PATH", "/opt/rocm") + "/llvm/bin") or shutil.which("llvm-readelf")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Template arguments (type, KH, RC, ONE, ANY, FW) -> what the code object says of the kernel"""
    if READELF is None:
        pytest.skip("no llvm-readelf")
    with open(_lib.LIB_PATH, "rb") as f:
        objects = [o for o in _code_objects(f.read()) if b"row_few_kernel" in o]
    assert len(objects) == 1
    path = tmp_path_factory.mktemp("few") / "code.o"
    path.write_bytes(objects[0])
    text = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
    found = {}
    for entry in re.split(r"\n  - ", text):
        name = re.search(r"row_few_kernelI(DF16b?|DF16_)Li(\d)ELi\d+ELi(\d+)ELi\d+ELb([01])ELb([01])ELi(\d)E", entry)
        if name and "private_segment_fixed_size" in entry:
            key = (name[1],) + tuple(int(v) for v in name.groups()[1:])
            found[key] = {k: int(v) for k, v in re.findall(r"\.(vgpr_count|private_segment_fixed_size|vgpr_spill_count): +(\d+)", entry)}
    assert len(found) == 32          # 3x3: eight of each type, 5x5 and 7x7 four
    return found


def test_nothing_goes_to_scratch_memory(kernels):
    assert {k: v for k, v in kernels.items() if v["private_segment_fixed_size"] or v["vgpr_spill_count"]} == {}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K,block,scattered", [
    ((1, 512, 7, 7), 512, 1, 0), ((1, 512, 7, 7), 320, 0, 0), ((1, 512, 7, 7), 128, 0, 0), ((1, 288, 10, 10), 320, 1, 0), ((1, 288, 10, 10), 256, 0, 0),
    ((1, 1024, 7, 7), 640, 0, 0),                                                                 # more than an item to a pair of wavefronts
    ((1, 256, 14, 14), 256, 1, 1), ((2, 160, 24, 27), 160, 1, 1), ((8, 160, 14, 14), 160, 0, 0),    # eight; five, 210 and 280 workgroups
    ((8, 128, 14, 14), 160, 1, 1), ((16, 128, 14, 14), 160, 0, 0), ((4, 96, 20, 20), 256, 1, 1), ((16, 96, 12, 12), 256, 0, 0),      # four, 280 and 560; three, 448 and 768
    ((8, 32, 24, 24), 160, 1, 1), ((8, 64, 24, 24), 128, 1, 1),                                   # one, 720; two, 576
])
def test_filters_taken_as_they_are(dtype, xs, K, block, scattered):
    """Where one launch was the faster call: taps in blocks of eight channels, and scattered ones as an input gradient's."""
    d = engine.make_desc(xs, (K, xs[1], 3, 3), dtype, 1, 1, 4, stacked=None, row=True)
    assert d.row == 1
    strides = {"block": (xs[1] * 9, 9, 0, 3, 1), "scattered": (9, K * 9, 0, -3, -1)}
    takes = {}
    for name, s in strides.items():
        found = ctypes.c_int(-1)
        _lib.check(_lib.load().wc_conv_takes_filter(ctypes.byref(d), ctypes.c_void_p(1 << 20), (ctypes.c_int64 * 5)(*s), ctypes.byref(found)))
        takes[name] = found.value
    assert takes == {"block": block, "scattered": scattered}
