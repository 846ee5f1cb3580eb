"""The row form's kernel for few tiles (conv_row_few.hip) keeps what it works on in registers: looked up in the built code."""
import os
import re
import shutil
import subprocess

import pytest

from pytorch_winoconv_amd import _lib
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
    assert len(found) >= 32
    return found


def test_nothing_goes_to_scratch_memory(kernels):
    assert {k: v for k, v in kernels.items() if v["private_segment_fixed_size"] or v["vgpr_spill_count"]} == {}
