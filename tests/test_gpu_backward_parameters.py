"""Weight and bias gradient in one call (wc_conv_backward_parameters): the column sums of dy that the kernels take on the way.

Exact on small integers: every form (tap form through registers and by LDS-DMA, one and two groups of output channels, direct products of
strided and 1x1 layers, transform domain, fp32), a last part that is nearly empty, fewer steps than turns, channels that fill little of
a tile, both result types and both host layers.  The reference has no backward pass (src/back/utils.cu:15-24)."""
import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad
    ((2, 40, 9, 11), (24, 40, 3, 3), 1, 1), ((1, 8, 3, 3), (8, 8, 3, 3), 1, 1), ((3, 64, 30, 31), (136, 64, 3, 3), 1, 1),
    ((2, 136, 21, 17), (192, 136, 3, 3), 1, (0, 1)), ((2, 50, 19, 18), (70, 50, 3, 3), 1, 1), ((1, 24, 5, 6, 7), (72, 24, 3, 3, 3), 1, 1),
    ((9, 64, 28, 28), (128, 64, 3, 3), 1, 1),
    ((2, 32, 33, 31), (40, 32, 3, 3), 2, 1), ((3, 136, 20, 24), (200, 136, 3, 3), 2, 1), ((40, 72, 9, 9), (72, 72, 5, 5), 2, 2),
    ((3, 32, 17, 19), (40, 32, 1, 1), 1, 0), ((5, 136, 40, 40), (264, 136, 1, 1), 1, 0), ((2, 16, 12, 12), (8, 16, 7, 7), 1, 3), ((2, 5, 9, 11), (7, 5, 4, 3), 1, (1, 0)),
]


@pytest.mark.parametrize("ext", [True, False])
@pytest.mark.parametrize("dtype,own", [(torch.float16, torch.float16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("case", CASES)
def test_bias_gradient_is_exact_and_the_weight_gradient_unchanged(dev, monkeypatch, case, dtype, own, ext):
    xs, ws, stride, pad = case
    monkeypatch.setattr(engine, "USE_EXT", ext)
    nd = len(xs) - 2
    fmt = torch.channels_last if nd == 2 else torch.channels_last_3d
    g = torch.Generator().manual_seed(5)
    conv = torch.nn.functional.conv2d if nd == 2 else torch.nn.functional.conv3d
    x, w = torch.randint(-2, 3, xs, generator=g).double(), torch.zeros(ws, dtype=torch.float64)
    y = conv(x, w, None, stride, pad)
    dy = torch.randint(0, 2, y.shape, generator=g).double() * (torch.arange(ws[0]).view([1, -1] + [1] * nd) % 5 - 2)    # channels differ
    xd, dyd = (t.to(dtype).to(dev).contiguous(memory_format=fmt) for t in (x, dy))
    dw, db = engine.conv_backward_parameters(xd, dyd, ws, stride, pad, 2, True, own, own)
    assert dw.dtype == db.dtype == own and torch.equal(db.cpu().double(), dy.sum([0] + list(range(2, nd + 2))).to(own).double())
    plain = engine.conv_backward_weight(xd, dyd, ws, stride, pad, 2)
    assert torch.equal(dw.to(dtype), plain)
    assert engine.conv_backward_parameters(xd, dyd, ws, stride, pad, 2, False, own)[1] is None


def test_what_is_refused(dev):
    x, dy = torch.randn(2, 8, 6, 6, device=dev).half(), torch.randn(2, 8, 6, 6, device=dev).half()
    with pytest.raises(ValueError):
        engine.conv_backward_parameters(x, dy[:, :, :5], (8, 8, 3, 3), 1, 1)
    with pytest.raises(TypeError):
        engine.conv_backward_parameters(x, dy.float(), (8, 8, 3, 3), 1, 1)
    with pytest.raises(ValueError):
        engine.conv_backward_parameters(x[:0], dy[:0], (8, 8, 3, 3), 1, 1)
    dw, db = engine.conv_backward_parameters(x, dy, (8, 8, 3, 3), 1, 1, 2, True, torch.float32, torch.float64)
    assert dw.dtype == torch.float32 and db.dtype == torch.float64
