"""The weight gradient of strided and one-tap layers taken directly (gemm_tn.hip), operands by LDS-DMA and through registers, and the
sum of its parts on the way to dw.

Integers whose sums stay below 2^24 are exact in fp32, so only the last rounding remains, the same on both sides.  NaN stands around x and
dy in memory, which rows past a part's end and pixels outside the image must not read."""

import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad
    ((1, 8, 3, 3), (8, 8, 3, 3), 2, 1), ((1, 8, 1, 1), (16, 8, 1, 1), 1, 0),                 # fewer stages than loads in flight
    ((2, 72, 11, 9), (136, 72, 3, 3), 2, 1), ((3, 64, 12, 7), (64, 64, 1, 1), 1, 0),         # last rows and columns of both tiles
    ((40, 16, 2, 3), (24, 16, 3, 3), 2, 1),                                                  # many small images in a stage
    ((2, 136, 31, 37), (72, 136, 5, 2), 2, (2, 0)), ((8, 128, 30, 30), (136, 128, 1, 1), 1, 0),   # several parts, the last one short
    ((9, 128, 70, 66), (128, 128, 3, 3), 2, 1),                                              # more than L2 holds: taps as neighbours
]


@pytest.mark.parametrize("shift", [0, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", CASES)
def test_exact_on_small_integers(dev, dtype, case, shift):
    """shift: tensors that start 8 or 16 bytes past a multiple of 16 (16-bit: through registers); the filter gradient through both
    memory orders."""
    xs, ws, stride, pad = case
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-3, 4, xs, generator=g).double()
    y = torch.nn.functional.conv2d(x[:1], torch.zeros(ws, dtype=torch.double), None, stride, pad)
    dy = torch.randint(-3, 4, (xs[0],) + tuple(y.shape[1:]), generator=g).double()
    want = torch.nn.grad.conv2d_weight(x, ws, dy, stride, pad).float().to(dtype)

    def guarded(t):
        flat = torch.full((t.numel() + 4096,), float("nan"), dtype=dtype, device=dev)[2048 + shift:2048 + shift + t.numel()]
        last = t.to(dev).to(dtype).movedim(1, -1)
        return flat.view(last.shape).copy_(last).movedim(-1, 1)

    dw = engine.conv_backward_weight(guarded(x), guarded(dy), ws, stride, pad, 2)
    assert torch.equal(dw.cpu(), want)
