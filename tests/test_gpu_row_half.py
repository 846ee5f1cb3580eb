"""Row form, 5x5: layers that 64-tile boxes cover in one round and 32-tile ones in two (make_row_shape in conv_row.hip), where that ends: the
bound of test_gpu_row_5x5_7x7.py."""
import pytest
import torch
import torch.nn.functional as F

from pytorch_winoconv_amd import engine
from test_gpu_row import _err, _row
from test_gpu_row_5x5_7x7 import BOUND, _operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K,pad", [
    ((37, 256, 13, 8), 203, 2), ((13, 199, 19, 19), 188, 2), ((5, 256, 42, 42), 65, 2),      # ragged channels, output channels and boxes
    ((64, 256, 8, 10), 256, 2), ((65, 256, 8, 10), 256, 2), ((65, 193, 9, 10), 256, (1, 2)),  # 256 boxes of 64 tiles (512 of 32) and the first beyond
])
def test_one_round_of_half_boxes_against_fp64(dev, dtype, xs, K, pad, gemm_override):
    x, w, b = _operands(xs, K, dtype)
    ref = F.conv2d(x.double(), w.double(), b.double(), padding=pad)
    assert engine.make_desc(xs, w.shape, dtype, 1, pad, 2, stacked=None, row=True).row == 1
    y = _row(x.to(dev), w.to(dev), b.to(dev), pad)
    assert _err(y, ref) <= BOUND[dtype]
    gemm_override(config=17)
    assert torch.equal(_row(x.to(dev), w.to(dev), b.to(dev), pad), y)      # either shape sums the channels in one order
