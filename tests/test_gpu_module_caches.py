"""What the modules keep between passes: the transformed filter and the plan of the last shape.  The reference keeps nothing
(conv.py:324-339)."""
import pytest
import torch
import torch.nn.functional as F

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu


def _input(dev, *shape, dtype=torch.float16, seed=1):
    x = torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(dev)
    return x.contiguous(memory_format=torch.channels_last if x.dim() == 4 else torch.channels_last_3d)


def _close(y, layer, x):
    want = F.conv2d(x.double(), layer.weight.double(), None if layer.bias is None else layer.bias.double(), layer.stride, layer.padding)
    assert y.dtype == x.dtype and (y.double() - want).norm() <= (1e-5 if x.dtype == torch.float32 else 1e-2) * want.norm()


def test_a_renewed_filter_is_kept_for_what_it_was_made_for(dev, monkeypatch):
    """A pass of another type, past the plan, between the planned pass that made the filter and the one that renews it (another thread's
    would do the same): the renewed filter is not taken for one of the other type."""
    layer = pkg.WinoConv2d(40, 24, 3, padding=1, device=dev).requires_grad_(False)
    half, single = _input(dev, 2, 40, 9, 11), _input(dev, 2, 40, 9, 11, dtype=torch.float32)
    for _ in range(3):
        layer(half)
    assert layer._plan[1] is not None
    monkeypatch.setattr(engine, "USE_EXT", False)
    _close(layer(single), layer, single)
    layer.weight.mul_(2)
    monkeypatch.setattr(engine, "USE_EXT", True)
    _close(layer(half), layer, half)
    monkeypatch.setattr(engine, "USE_EXT", False)
    _close(layer(single), layer, single)
    _close(layer(half), layer, half)


class _Counted(torch.nn.Module):
    """A parametrization with state, like a spectral norm's power iteration."""

    def __init__(self):
        super().__init__()
        self.calls = 0

    def forward(self, w):
        self.calls += 1
        return w * 1.0


def test_parameters_are_read_once_in_a_pass(dev):
    layer = pkg.WinoConv2d(16, 24, 3, padding=1, device=dev, dtype=torch.float16)
    counted = {}
    for name in ("weight", "bias"):
        torch.nn.utils.parametrize.register_parametrization(layer, name, _Counted())
        counted[name] = layer.parametrizations[name][0]
    shapes = [(2, 16, 9, 11)] * 4 + [(1, 16, 9, 11), (2, 16, 9, 11), (2, 16, 8, 11), (2, 16, 9, 11), (2, 16, 9, 11), (2, 16, 9, 11)]
    for i, shape in enumerate(shapes):
        before = counted["weight"].calls, counted["bias"].calls
        layer(_input(dev, *shape) if i % 3 else _input(dev, *shape).contiguous())
        assert (counted["weight"].calls, counted["bias"].calls) == (before[0] + 1, before[1] + 1), i


def test_hyperparameters_that_change_in_place(dev):
    layer = pkg.WinoConv2d(16, 24, 3, padding=1, device=dev, dtype=torch.float16).requires_grad_(False)
    layer.padding = [1, 1]
    x = _input(dev, 2, 16, 9, 11)
    for _ in range(4):
        _close(layer(x), layer, x)
    layer.padding[0] = 0
    assert layer(x).shape == (2, 24, 7, 11)
    _close(layer(x), layer, x)
