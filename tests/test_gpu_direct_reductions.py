"""The direct form over short and long reductions (gemm_kernel<..., DIRECT>: loads one or two reduction blocks ahead) on each
tile that it chooses between.  A convolution in fp64 pins it (the reference refuses stride 2: src/winograd_conv.cpp:122-126).

Bound: exact operands, fp32 sums, one rounding of the result: 2^-p relative for p bits of significand, plus 1e-5 of the
2-norm for the sums."""
import pytest
import torch
import torch.nn.functional as F

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu
BOUND = {torch.float32: 1e-5, torch.float16: 2.0 ** -11 + 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5}

CASES = [
    # x shape, K, kernel, stride: reduction blocks of 32
    ((1, 32, 5, 6), 8, 1, 1), ((2, 64, 7, 5), 72, 1, 1), ((2, 96, 9, 9), 40, 1, 1),       # 1, 2 and 3
    ((1, 32, 9, 8), 24, 3, 2), ((3, 64, 15, 14), 72, 3, 2),                               # 9 and 18, small tiles
    ((12, 64, 111, 113), 136, 3, 2), ((10, 32, 80, 81), 72, 1, 1),                        # 128 x 128 tiles
    ((22, 96, 113, 111), 72, 3, 2),                                                       # 256 x 128
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_against_fp64(dev, dtype, case):
    xs, K, k, stride = case
    g = torch.Generator().manual_seed(9)
    x = torch.randn(xs, generator=g).to(dtype)
    w = (torch.randn((K, xs[1], k, k), generator=g) * 0.1).to(dtype)
    ref = F.conv2d(x.double(), w.double(), stride=stride, padding=k // 2)
    x = x.to(dev).contiguous(memory_format=torch.channels_last)
    y = engine.conv_forward(x, w.to(dev), None, stride, k // 2, 2, direct=True)
    assert float((y.double().cpu() - ref).norm() / ref.norm()) <= BOUND[dtype]
