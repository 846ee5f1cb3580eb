"""The row form's tall boxes (conv_row_tall.hip): the bound and the operands of test_gpu_row.py, which pins the tile itself."""
import pytest
import torch

from pytorch_winoconv_amd import engine
from test_gpu_row import BOUND, CASES, _conv64, _err, _operands, _row

pytestmark = pytest.mark.gpu

EDGES = [
    ((1, 32, 4, 128), 128, 1), ((33, 40, 5, 4), 128, 1),              # 32 columns in one row; one column more, one row more
    ((2, 8, 1, 260), 136, (1, 1)), ((31, 72, 9, 6), 8, 0),            # columns across images; one block of channels and 8 more
    ((2, 64, 2, 3, 130), 129, 1), ((7, 96, 4, 6, 9), 40, (0, 1, 1)),  # tap planes beyond either end
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES[2:] + EDGES)
def test_against_fp64(dev, dtype, case, gemm_override):
    xs, K, pad = case
    x, w, b = _operands(xs, K, dtype)
    gemm_override(config=21)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), _conv64(x, w, b, pad)) <= BOUND[dtype]
    assert _err(_row(x.to(dev), w.to(dev), None, pad), _conv64(x, w, None, pad)) <= BOUND[dtype]


@pytest.mark.parametrize("xs,K", [((67, 64, 54, 60), 136), ((9, 40, 14, 50, 52), 129)])
def test_several_boxes_a_workgroup(dev, xs, K, gemm_override):
    """More boxes than CUs, the last of them partial; workgroups with one box more than others."""
    x, w, b = _operands(xs, K, torch.float16)
    gemm_override(config=21)
    y = _row(x.to(dev), w.to(dev), b.to(dev), 1)
    assert _err(y, _conv64(x, w, b, 1)) <= BOUND[torch.float16]
    assert torch.equal(_row(x.to(dev), w.to(dev), b.to(dev), 1), y)


def test_batch_cut_in_tall_boxes_and_others(dev, gemm_override):
    """61 of 64 images fill three rounds of tall boxes, the rest takes another shape: each image has the bits of its shape, also
    where the batch comes in passes that do not end at the cut."""
    x, w, b = _operands((64, 160, 56, 56), 256, torch.float16)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    y = _row(xd, wd, bd, 1)
    ref = torch.nn.functional.conv2d(x[58:].double(), w.double(), b.double(), padding=1)
    assert _err(y[58:], ref) <= BOUND[x.dtype]
    passes = engine.conv_forward(xd, wd, bd, 1, 1, 2, chunk_images=27, row=True)
    gemm_override(config=21)
    tall = _row(xd, wd, bd, 1)
    assert torch.equal(y[:61], tall[:61]) and not torch.equal(y[61:], tall[61:])
    assert torch.equal(passes, y)


def test_batch_cut_within_the_last_image(dev, gemm_override):
    """756 tall boxes hold 123 of 128 output planes; the other five, all of the last image, take another shape."""
    x, w, b = _operands((8, 64, 16, 56, 56), 128, torch.float16)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    y = _row(xd, wd, bd, 1)
    ref = torch.nn.functional.conv3d(x[7:, :, 9:].double(), w.double(), b.double(), padding=1)[:, :, 1:]
    assert _err(y[7:, :, 10:], ref) <= BOUND[x.dtype]
    passes = engine.conv_forward(xd, wd, bd, 1, 1, 2, chunk_images=3, row=True)
    gemm_override(config=21)
    tall = _row(xd, wd, bd, 1)
    assert torch.equal(y[:7], tall[:7]) and torch.equal(y[7, :, :11], tall[7, :, :11]) and not torch.equal(y[7, :, 11:], tall[7, :, 11:])
    assert torch.equal(passes, y)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K", [((3, 40, 9, 30), 136), ((2, 32, 3, 5, 18), 64)])
def test_bias_that_starts_anywhere(dev, dtype, xs, K, gemm_override, host_layer):
    """A bias that is a view into a flat buffer gives the bits of an aligned one: the same values are added."""
    x, w, b = _operands(xs, K, dtype)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    gemm_override(config=21)
    want = _row(xd, wd, bd, 1)
    assert _err(want, _conv64(x, w, b, 1)) <= BOUND[dtype]
    layer = engine.conv_forward(xd, wd, bd, 1, 1, 2, row=True)
    for first in (1, 2, 3, 4, 7):
        view = torch.full((K + 16,), float("nan"), dtype=dtype, device=dev)[first:first + K].copy_(bd)
        assert view.data_ptr() % 16 == 2 * first
        assert torch.equal(_row(xd, wd, view, 1), want)
        assert torch.equal(engine.conv_forward(xd, wd, view, 1, 1, 2, row=True), layer)
