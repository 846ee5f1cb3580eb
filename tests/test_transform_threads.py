"""How the transforms of small 2-D plans share their work out (csrc/transform_threads.h): the line lies where both sides were measured."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pytorch_winoconv_amd", "csrc")
CXX = shutil.which("g++") or shutil.which("c++")


def _rows(tmp_path, call, rows):
    if CXX is None:
        pytest.skip("no C++ compiler")
    source, program = tmp_path / "t.cpp", tmp_path / "t"
    lines = "".join("  std::printf(\"%%d\\n\", (int)wc::%s(%s));\n" % (call, ", ".join(str(v).lower() for v in r)) for r in rows)
    source.write_text('#include <cstdio>\n#include "transform_threads.h"\nint main() {\n%s}\n' % lines)
    subprocess.run([CXX, "-std=c++17", "-I", CSRC, str(source), "-o", str(program)], check=True)
    return [int(v) for v in subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split()]


def test_channels_of_an_input_transform(tmp_path):
    """(channels at most, tiles, channels of a row, pieces, stacked, fp32, tile) -> channels"""
    cases = [
        ((4, 1125, 32, 4, True, True, 2), 4), ((4, 425, 96, 4, True, True, 2), 4), ((4, 216, 160, 4, True, True, 2), 4), ((4, 500, 160, 4, True, True, 2), 4),
        ((4, 512, 64, 9, True, True, 2), 4), ((4, 225, 64, 4, True, True, 2), 1), ((4, 64, 64, 9, True, True, 2), 1), ((4, 252, 128, 4, True, True, 2), 2),
        ((8, 225, 64, 4, True, False, 2), 1), ((8, 500, 160, 4, True, False, 2), 4), ((8, 288, 320, 4, True, False, 2), 4),
        ((2, 250, 128, 4, True, True, 4), 1), ((2, 250, 128, 4, True, False, 4), 1), ((2, 100, 128, 4, True, False, 4), 1),
        ((4, 484, 128, 4, False, True, 2), 2), ((4, 361, 64, 9, False, True, 2), 2), ((2, 225, 96, 4, False, False, 4), 1),
        ((1, 4, 32, 4, True, True, 2), 1), ((8, 100000, 512, 9, True, False, 2), 8),
    ]
    assert _rows(tmp_path, "input_channels", [c[0] for c in cases]) == [c[1] for c in cases]


def test_pieces_of_an_input_transform_apart(tmp_path):
    """(threads, pieces, stacked, fp32, tile) -> threads of its own for every piece"""
    cases = [
        ((158184, 4, False, False, 2), 1), ((186984, 4, False, False, 2), 0), ((258048, 4, False, False, 2), 0), ((199920, 4, False, False, 4), 1),
        ((368640, 4, False, False, 4), 0), ((457776, 4, False, False, 4), 0), ((258720, 9, False, False, 2), 1), ((460800, 9, False, False, 4), 1),
        ((492840, 4, False, True, 2), 1), ((460800, 9, False, True, 4), 1), ((802816, 9, False, True, 2), 0), ((500000, 4, True, False, 2), 1), ((600000, 9, True, True, 4), 0),
    ]
    assert _rows(tmp_path, "pieces_apart", [c[0] for c in cases]) == [c[1] for c in cases]


def test_channels_of_an_output_transform(tmp_path):
    """(tiles, output channels, channels at most, pieces, fp32, tile) -> one channel a thread"""
    cases = [
        ((784, 136, 2, 1, False, 4), 0), ((1600, 64, 2, 1, False, 4), 0), ((480, 112, 2, 1, False, 4), 1), ((784, 136, 2, 1, True, 4), 1), ((1800, 64, 2, 1, True, 4), 1),
        ((972, 216, 4, 1, True, 2), 0), ((972, 216, 4, 1, False, 2), 0), ((841, 64, 4, 1, False, 2), 1), ((3072, 56, 4, 4, True, 2), 1), ((2000, 40, 2, 4, False, 4), 1),
        ((4000, 40, 2, 4, False, 4), 0), ((4000, 40, 2, 1, True, 4), 0),
    ]
    assert _rows(tmp_path, "output_one_channel", [c[0] for c in cases]) == [c[1] for c in cases]
