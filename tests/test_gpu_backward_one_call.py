"""A module's backward pass in one call of the compiled host layer (engine.conv_backward) against the gradient functions one by
one, through ctypes: the same kernels, so the same bits.  The reference has no backward pass (src/back/utils.cu:15-24)."""
import pytest
import torch

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

LAYERS = [
    # module, x shape, out channels, kernel, stride, padding
    (pkg.WinoConv2d, (2, 40, 9, 11), 24, 3, 1, 1), (pkg.WinoConv2d, (2, 256, 9, 8), 64, 3, 1, 1), (pkg.WinoConv2d, (2, 16, 12, 13), 44, 5, 1, 2),
    (pkg.WinoConv2d, (2, 32, 15, 14), 32, 3, 2, 1), (pkg.WinoConv2d, (1, 20, 10, 9), 12, 4, 2, 1),      # without and with zeros between dy
    (pkg.WinoConv3d, (1, 24, 5, 6, 7), 40, 3, 1, 1), (pkg.WinoConv3d, (1, 16, 6, 7, 6), 16, 3, 2, 1),
]


def _layer(dev, case, dtype, own):
    kind, xs, K, taps, stride, pad = case
    torch.manual_seed(4)
    layer = kind(xs[1], K, taps, stride=stride, padding=pad, device=dev, dtype=own)
    with torch.no_grad():
        layer.bias.normal_()
    fmt = torch.channels_last if len(xs) == 4 else torch.channels_last_3d
    return layer, torch.randn(xs, device=dev).to(dtype).contiguous(memory_format=fmt).requires_grad_(True)


@pytest.mark.parametrize("dtype,own", [(torch.float16, torch.float16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                       (torch.float32, torch.float32)])
@pytest.mark.parametrize("case", LAYERS)
def test_same_as_one_by_one(dev, monkeypatch, case, dtype, own):
    layer, x = _layer(dev, case, dtype, own)
    params = (x, layer.weight, layer.bias)

    def gradients(wanted, dy):
        y = layer(x)
        return torch.autograd.grad(y, [params[i] for i in wanted], torch.randn(y.shape, device=dev, generator=torch.Generator(dev).manual_seed(1))
                                   .to(dtype).contiguous(memory_format=dy))

    fmt = torch.channels_last if x.dim() == 4 else torch.channels_last_3d
    for wanted in ((0, 1, 2), (1, 2), (0,), (2,)):
        for dy in (fmt, torch.contiguous_format):
            monkeypatch.setattr(engine, "USE_EXT", True)
            got = gradients(wanted, dy)
            monkeypatch.setattr(engine, "USE_EXT", False)
            for a, b, i in zip(got, gradients(wanted, dy), wanted):
                assert a.dtype == params[i].dtype and a.shape == params[i].shape and torch.equal(a, b), (wanted, i)


def test_hooks_graphs_and_what_is_refused(dev):
    """Saved-tensor hooks see x and the filter; a dy that is one value expanded; a graph of the gradients; a parameter without
    gradient; function transforms stay refused."""
    layer, x = _layer(dev, LAYERS[0], torch.float16, torch.float32)
    y = layer(x)
    want = torch.autograd.grad(y, (x, layer.weight, layer.bias), torch.ones_like(y))
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1], lambda t: t.to(dev)):
        y = layer(x)
    got = torch.autograd.grad(y, (x, layer.weight, layer.bias), torch.ones_like(y))
    assert sorted(seen) == sorted([x.shape, layer.weight.shape]) and all(torch.equal(a, b) for a, b in zip(got, want))
    layer(x).sum().backward()                                    # dy is one value
    assert torch.equal(x.grad, want[0]) and torch.equal(layer.weight.grad, want[1]) and torch.allclose(layer.bias.grad, want[2])
    dy = torch.ones_like(y).requires_grad_(True)
    db = torch.autograd.grad(layer(x), layer.bias, dy, create_graph=True)[0]
    assert torch.equal(torch.autograd.grad(db.sum(), dy)[0], torch.ones_like(dy))
    layer.bias.requires_grad_(False)
    assert torch.equal(torch.autograd.grad(layer(x), layer.weight, torch.ones_like(y))[0], want[1])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: layer(t).float().sum())(x.detach())
