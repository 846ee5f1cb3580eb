"""The fp32 weight gradient on 2-D plans of tile 4: its product takes three bf16 parts per operand (gemm_tn.hip) where the fp32
instructions, forced here, round more.  Both against fp64: the bound is the error of the fp32 instructions itself, with a tenth for the
spread of a sum of few values."""

import pytest
import torch
import torch.nn.functional as F

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,k,h,w,taps", [
    (1, 8, 8, 4, 4, 3), (2, 40, 72, 17, 19, 3), (4, 64, 64, 28, 28, 3), (8, 136, 200, 30, 26, 3),   # one tile; both tile sizes; several parts
    (3, 72, 65, 9, 40, 3), (2, 32, 96, 21, 20, 5),
])
def test_no_larger_error_than_the_fp32_instructions(dev, n, c, k, h, w, taps, gemm_override):
    g = torch.Generator().manual_seed(7)
    x = torch.randn(n, c, h, w, generator=g)
    dy = torch.randn(n, k, h, w, generator=g)
    shape = (k, c, taps, taps)
    ref = torch.nn.grad.conv2d_weight(x.double(), shape, dy.double(), 1, taps // 2)

    def err():
        dw = engine.conv_backward_weight(x.to(dev), dy.to(dev), shape, 1, taps // 2, 4)
        return float((dw.cpu().double() - ref).norm() / ref.norm())

    split = err()
    gemm_override(config=22)
    assert split <= 1.1 * err()


def test_long_sums_of_one_sign(dev, gemm_override):
    """Parts of some thousand tiles, x and dy without negative values, 32 of the input channels against fp64."""
    n, c, h = 64, 256, 56
    g = torch.Generator(device=dev).manual_seed(7)
    x, dy = torch.randn(n, c, h, h, generator=g, device=dev).relu(), torch.randn(n, c, h, h, generator=g, device=dev).abs()
    ref = torch.zeros(c, 32, 3, 3, dtype=torch.float64, device=dev)
    for a in range(0, n, 8):
        xp = F.pad(x[a:a + 8, :32].double(), [1] * 4)
        d = dy[a:a + 8].double().movedim(1, -1).reshape(-1, c).t().contiguous()
        for i in range(3):
            for j in range(3):
                ref[:, :, i, j] += d @ xp[:, :, i:i + h, j:j + h].movedim(1, -1).reshape(-1, 32).contiguous()
    x, dy = (t.contiguous(memory_format=torch.channels_last) for t in (x, dy))

    def err():
        dw = engine.conv_backward_weight(x, dy, (c, c, 3, 3), 1, 1, 4)[:, :32]
        return float((dw.double() - ref).norm() / ref.norm())

    split = err()
    gemm_override(config=22)
    assert split <= 1.1 * err()


def test_an_infinity_stays_out_of_other_channels(dev):
    x = torch.randn(2, 40, 12, 12)
    dy = torch.randn(2, 72, 12, 12)
    x[1, 7, 5, 5] = float("inf")
    dw = engine.conv_backward_weight(x.to(dev), dy.to(dev), (72, 40, 3, 3), 1, 1, 4).cpu()
    assert not torch.isfinite(dw[:, 7]).any()
    assert torch.isfinite(dw[:, :7]).all() and torch.isfinite(dw[:, 8:]).all()
