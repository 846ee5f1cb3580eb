"""The row form on boxes of few tiles (conv_row_few.hip): the bounds of test_gpu_row.py and test_gpu_row_5x5_7x7.py, where workgroups, pairs of
wavefronts and their items end."""
import pytest
import torch
import torch.nn.functional as F

import test_gpu_row as three
import test_gpu_row_5x5_7x7 as more
from pytorch_winoconv_amd import engine
from test_gpu_row import _err, _row

pytestmark = pytest.mark.gpu

EDGES = [
    ((1, 32, 7, 7), 8, 1), ((1, 32, 7, 7), 9, 1), ((2, 8, 5, 6), 40, 1), ((2, 8, 5, 6), 41, 1),       # output channels: a block's second sixteen rows
    ((1, 256, 6, 9), 32, 1), ((1, 257, 6, 9), 32, 1), ((1, 520, 4, 7), 24, 1),                      # items: eight pairs with one each; nine; five to some
    ((17, 96, 4, 4), 48, 1), ((1, 64, 33, 70), 16, 0),                                             # boxes of images; many boxes
    ((1, 65, 3, 7, 5), 33, 1), ((2, 96, 4, 6, 7), 16, (1, 0, 1)),                                   # items of planes of taps: nine
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", three.CASES + EDGES)
def test_3x3_and_3x3x3_against_fp64(dev, dtype, case, gemm_override):
    xs, K, pad = case
    x, w, b = three._operands(xs, K, dtype)
    gemm_override(config=30)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), three._conv64(x, w, b, pad)) <= three.BOUND[dtype]
    assert _err(_row(x.to(dev), w.to(dev), None, pad), three._conv64(x, w, None, pad)) <= three.BOUND[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("taps,case", [(5, c) for c in more.CASES + [((1, 256, 7, 7), 40, 2), ((1, 264, 5, 9), 9, 2)]] +
                         [(7, c) for c in more.CASES_7 + [((1, 128, 9, 9), 40, 3), ((1, 129, 7, 8), 9, 3)]])
def test_5x5_and_7x7_against_fp64(dev, dtype, taps, case, gemm_override):
    xs, K, pad = case
    x, w, b = more._operands(xs, K, dtype, taps=taps)
    gemm_override(config=30)
    ref = F.conv2d(x.double(), w.double(), b.double(), padding=pad)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), ref) <= more.BOUND[dtype]


@pytest.mark.parametrize("xs,K", [((1, 512, 7, 7), 512), ((3, 160, 14, 13), 96), ((2, 129, 9, 9), 200), ((2, 72, 3, 6, 7), 40)])
def test_chosen_and_in_passes(dev, xs, K, gemm_override):
    """The library's choice is this kernel, bit for bit, for a whole batch and image by image."""
    x, w, b = (t.to(dev) for t in three._operands(xs, K, torch.float16))
    d = engine.make_desc(xs, w.shape, x.dtype, 1, 1, 2, stacked=None, row=True)
    assert d.row == 1
    y = engine.conv_forward(x, w, b, 1, 1, 2, row=True)
    assert torch.equal(engine.conv_forward(x, w, b, 1, 1, 2, chunk_images=1, row=True), y)
    gemm_override(config=30)
    assert torch.equal(engine.conv_forward(x, w, b, 1, 1, 2, row=True), y)
