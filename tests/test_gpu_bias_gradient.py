"""The bias gradient (bias_gradient.hip).  The reference has no backward pass (src/back/utils.cu:15-24); a sum in fp64 pins it.

Bound: fp32 sums of n values, at most n 2^-24 of the sum of magnitudes (the sums are split, so far below it: 1e-6 of it here)
and the rounding of the result, 2^-p relative."""
import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu
EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}

SHAPES = [(1, 1, 1, 1), (1, 8, 1, 1), (2, 3, 5, 7), (3, 100, 9, 11), (2, 150, 7, 5), (3, 24, 9, 11), (2, 264, 13, 6), (1, 2056, 3, 5), (1, 600, 31, 33),
          (5, 128, 40, 41), (64, 64, 56, 56), (2, 40, 3, 9, 10)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_against_fp64(dev, dtype, shape, shift):
    g = torch.Generator().manual_seed(7)
    last = torch.randn([shape[0]] + list(shape[2:]) + [shape[1]], generator=g).to(dtype)
    flat = torch.empty(last.numel() + 8, dtype=dtype, device=dev)[shift:shift + last.numel()]
    dy = flat.view(last.shape).copy_(last)                              # shift 1: rows that do not start at 16 bytes
    db = engine.bias_gradient(dy.permute([0, dy.dim() - 1] + list(range(1, dy.dim() - 1))))
    rows = last.double().reshape(-1, shape[1])
    ref, size = rows.sum(0), rows.abs().sum(0)
    assert db.shape == (shape[1],) and db.dtype == dtype
    assert bool(((db.double().cpu() - ref).abs() <= EPS[dtype] * ref.abs() + 1e-6 * size).all())


def test_channel_first_and_empty(dev):
    dy = torch.randn(3, 5, 4, 6, device=dev)
    assert torch.allclose(engine.bias_gradient(dy), dy.sum((0, 2, 3)), atol=1e-4)
    assert bool((engine.bias_gradient(dy[:0]) == 0).all())
