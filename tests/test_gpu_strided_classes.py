"""The input gradient of strided layers, all parity classes of its pixels in one product (gemm_direct_classes in gemm.hip).
The reference has no backward pass (src/back/utils.cu:15-24); the gradient of a convolution in fp64 pins it.

Bound: exact operands, fp32 sums, one rounding of the result: 2^-p relative for p bits of significand, plus 1e-5 of the
2-norm for the sums."""
import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu
BOUND = {torch.float32: 1e-5, torch.float16: 2.0 ** -11 + 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5}

CASES = [
    # x shape, K, kernel, pad
    ((1, 8, 3, 3), 32, (3, 3), 1), ((1, 8, 1, 5), 32, (3, 3), 1),      # one pixel of some classes, none of others
    ((2, 72, 15, 18), 32, (3, 3), 1), ((3, 136, 17, 13), 64, (5, 5), 2),   # classes of different sizes, channel remainders
    ((2, 16, 12, 9), 32, (2, 5), (0, 1)), ((2, 24, 9, 9), 32, (1, 3), (0, 1)),   # one tap on an axis: classes of zeros
    ((9, 96, 67, 65), 32, (3, 3), 1), ((24, 72, 75, 74), 32, (3, 3), 1),   # 128 x 128 and 256 x 128 tiles, partial edges
    ((1, 8, 20, 20), 32, (7, 7), 3),                                   # kernel rows of four taps: a launch per class
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_against_fp64(dev, dtype, case):
    xs, K, kernel, pad = case
    g = torch.Generator().manual_seed(5)
    pads = (pad, pad) if isinstance(pad, int) else pad
    w = (torch.randn((K, xs[1]) + kernel, generator=g) * 0.1).to(dtype)
    out = [(xs[2 + i] + 2 * pads[i] - kernel[i]) // 2 + 1 for i in range(2)]
    dy = torch.randn([xs[0], K] + out, generator=g).to(dtype)
    ref = torch.nn.grad.conv2d_input(xs, w.double(), dy.double(), stride=2, padding=pads)
    dx = engine.conv_backward_input(dy.to(dev), w.to(dev), xs[2:], 2, pads, 2)
    assert float((dx.double().cpu() - ref).norm() / ref.norm()) <= BOUND[dtype]
    assert bool((dx.cpu()[ref == 0] == 0).all())                       # classes that no tap reaches are zero, not left over
