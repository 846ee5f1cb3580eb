"""The fused F(2x2, 3x3) kernel on rows of 256 bytes (thin_rows_kernel in conv_thin.hip: 97 to 128 channels of a 16-bit type, 33 to 64 of fp32):
the exact integers of test_gpu_thin.py where its blocks, its rounds of blocks and its output channels end."""
import pytest
import torch
import torch.nn.functional as F

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

EDGES = [
    # N, C (16 bits; half as many in fp32), K, H, W, pad
    (1, 128, 64, 8, 8, 1), (1, 128, 64, 2, 34, 1),              # one block of 16 tiles; one tile more
    (1, 100, 3, 2, 2, 1), (2, 116, 61, 7, 5, 0),               # element-wise stores; half-used tiles
    (3, 128, 68, 9, 11, 1), (2, 124, 36, 10, 10, 2),           # a quad of output channels beyond 64; a group of 32 and a quad
    (2, 128, 128, 64, 64, 1), (2, 128, 128, 64, 66, 1),         # 128 blocks for 128 workgroups; some with two
    (3, 128, 256, 46, 64, 1), (9, 108, 200, 40, 44, 1),        # 64 workgroups of a group: two and three rounds, seven and a piece
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("config", [8, 9])
@pytest.mark.parametrize("shape", EDGES)
def test_exact_on_small_integers(dev, dtype, config, shape, gemm_override):
    """Both sizes of workgroup.  Every intermediate is an integer below 2^24, as in test_gpu_thin.py: 128 channels x 9 taps x 3 x 8 < 2^15 and at
    most 16 times that in a sum of transformed products."""
    N, C, K, H, W, pad = shape
    C = C // 2 if dtype == torch.float32 else C
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-3, 4, (N, C, H, W), generator=g).double()
    w = 4.0 * torch.randint(-2, 3, (K, C, 3, 3), generator=g).double()
    b = torch.randint(-8, 9, (K,), generator=g).double()
    gemm_override(config=config)
    for bias in (b, None):
        ref = F.conv2d(x.float(), w.float(), None if bias is None else bias.float(), padding=pad).to(dtype)
        y = engine.conv_forward(x.to(dtype).to(dev), w.to(dtype).to(dev), None if bias is None else bias.to(dtype).to(dev), 1, pad, 2)
        assert torch.equal(y.cpu(), ref)
