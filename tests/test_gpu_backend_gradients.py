"""The gradients through the compiled host layer (make_pytorch_backend.cpp) against the same calls through ctypes: one C ABI,
so the results are the same bit for bit.  The reference has no backward pass (src/back/utils.cu:15-24)."""
import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad
    ((2, 40, 9, 11), (24, 40, 3, 3), 1, 1), ((1, 24, 5, 6, 7), (40, 24, 3, 3, 3), 1, (0, 1, 1)),     # the row form's flipped filter
    ((2, 5, 9, 11), (7, 5, 4, 3), 1, (1, 0)), ((2, 8, 15, 14), (32, 8, 3, 3), 2, 1), ((2, 16, 12, 12), (8, 16, 7, 7), 1, 3),
    ((3, 32, 17, 19), (40, 32, 1, 1), 1, 0),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("last", [True, False])
@pytest.mark.parametrize("case", CASES)
def test_same_as_through_ctypes(dev, monkeypatch, dtype, last, case):
    xs, ws, stride, pad = case
    assert engine.USE_EXT
    g = torch.Generator().manual_seed(11)
    nd = len(xs) - 2
    pads = (pad,) * nd if isinstance(pad, int) else pad
    x = torch.randn(xs, generator=g).to(dtype).to(dev)
    w = torch.randn(ws, generator=g).to(dtype).to(dev)
    out = [(xs[2 + i] + 2 * pads[i] - ws[2 + i]) // stride + 1 for i in range(nd)]
    dy = torch.randn([xs[0], ws[0]] + out, generator=g).to(dtype).to(dev)
    if last:
        fmt = torch.channels_last if nd == 2 else torch.channels_last_3d
        x, dy, w = (t.contiguous(memory_format=fmt) for t in (x, dy, w))

    def gradients():
        return (engine.conv_backward_input(dy, w, xs[2:], stride, pad, 2), engine.conv_backward_weight(x, dy, ws, stride, pad, 2),
                engine.bias_gradient(dy))

    ours = gradients()
    monkeypatch.setattr(engine, "USE_EXT", False)
    for a, b in zip(ours, gradients()):
        assert a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def test_errors(dev):
    x, dy = torch.randn(2, 8, 6, 6, device=dev), torch.randn(2, 4, 6, 6, device=dev)
    with pytest.raises(TypeError):
        engine.conv_backward_weight(x, dy.half(), (4, 8, 3, 3), 1, 1)
    with pytest.raises(ValueError):
        engine.conv_backward_weight(x, dy[:, :, :5], (4, 8, 3, 3), 1, 1)
    with pytest.raises(ValueError):
        engine.conv_backward_weight(x, dy, (4, 7, 3, 3), 1, 1)
    with pytest.raises(NotImplementedError):
        engine.conv_backward_weight(x, dy, (4, 8, 3, 3), (1, 2), 1)
    with pytest.raises(ValueError):
        engine.bias_gradient(dy.cpu())
