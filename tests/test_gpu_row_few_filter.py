"""The row form on few tiles taking its filter as it is (conv_row_few.hip): the bits that a transformed filter gives, for every order of w that the kernel
takes, where output channels, blocks of channels and pairs of wavefronts end, and the same for those that it does not take."""
import ctypes

import pytest
import torch

from pytorch_winoconv_amd import WinoConv2d, _lib, engine

pytestmark = pytest.mark.gpu

SHAPES = [  # shape of x, output channels
    ((1, 8, 5, 6), 1), ((2, 32, 7, 7), 17), ((3, 40, 6, 9), 24), ((1, 72, 9, 9), 33), ((2, 256, 6, 5), 48),       # up to an item to a pair
    ((1, 264, 5, 7), 16), ((1, 512, 7, 7), 40),                                                               # more
]


def _orders(w):
    """w and tensors with the same values in other orders of memory, the last one not a kernel's"""
    K, C = w.shape[:2]
    turned = w.transpose(0, 1).contiguous().transpose(0, 1)
    odd = torch.empty(w.numel() + 1, dtype=w.dtype, device=w.device)[1:].view(w.shape)
    odd.copy_(w)
    wide = torch.empty(K, C, 9 + 5, dtype=w.dtype, device=w.device)[:, :, :9].view(K, C, 3, 3)
    wide.copy_(w)
    return [w, turned, odd, wide, w.contiguous(memory_format=torch.channels_last)]


def _takes(x, w):
    d = engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 4, stacked=None, row=True)
    takes = ctypes.c_int(-1)
    _lib.check(_lib.load().wc_conv_takes_filter(ctypes.byref(d), engine._ptr(w), engine._w_strides(w), ctypes.byref(takes)))
    return takes.value


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K", SHAPES)
def test_same_bits_as_a_transformed_filter(dev, dtype, xs, K, gemm_override):
    gemm_override(config=30)                      # few tiles, whatever the layer
    g = torch.Generator().manual_seed(K)
    x = torch.randn(xs, generator=g).to(dtype).to(dev).contiguous(memory_format=torch.channels_last)
    w = (torch.randn(K, xs[1], 3, 3, generator=g) * 0.1).to(dtype)
    w[K // 2, xs[1] // 2] = float("inf")          # reaches its own output channel only
    w, b = w.to(dev), torch.randn(K, generator=g).to(dtype).to(dev)
    U = engine.transform_filter(w, x.shape, 1, 1, 4, row=True)
    y = engine.conv_forward(x, w, b, 1, 1, 4, U=U, row=True)
    assert torch.isfinite(y.float()).all(dim=(0, 2, 3)).sum() >= K - 1
    orders = _orders(w)
    few = xs[1] <= 256
    assert [_takes(x, v) for v in orders] == [1, few, few, few, 0]
    for v in orders:
        assert torch.allclose(engine.conv_forward(x, v, b, 1, 1, 4, row=True).float(), y.float(), rtol=0, atol=0, equal_nan=True)
        assert torch.allclose(engine.conv_forward(x, v, b, 1, 1, 4, chunk_images=1, row=True).float(), y.float(), rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K", SHAPES)
def test_taps_against_the_order_of_memory(dev, dtype, xs, K, gemm_override):
    """An input gradient, whose filter is the layer's turned around, against the same convolution of a filter laid out that way."""
    gemm_override(config=30)
    g = torch.Generator().manual_seed(K + 1)
    dy = torch.randn(xs, generator=g).to(dtype).to(dev).contiguous(memory_format=torch.channels_last)
    w = (torch.randn(xs[1], K, 3, 3, generator=g) * 0.1).to(dtype).to(dev)      # of a layer K -> xs[1]
    turned = w.transpose(0, 1).flip(2, 3).contiguous()
    U = engine.transform_filter(turned, dy.shape, 1, 1, 4, row=True)
    ref = engine.conv_forward(dy, turned, None, 1, 1, 4, U=U, row=True)
    assert torch.equal(engine.conv_backward_input(dy, w, xs[2:], 1, 1, 4), ref)


def test_layers_of_channels_that_are_no_whole_chunks(dev):
    x = torch.randn(1, 36, 7, 7, device=dev, dtype=torch.float16).contiguous(memory_format=torch.channels_last)
    w = torch.randn(16, 36, 3, 3, device=dev, dtype=torch.float16)
    assert _takes(x, w) == 0
    assert _takes(x[:, :32], w[:, :32]) == 1 and _takes(x[:, :32].float(), w[:, :32].float()) == 0


@pytest.mark.parametrize("own", [torch.float16, torch.float32])
def test_module_passes_with_and_without_gradients(dev, own):
    """A weight that changes between passes is the one of its pass, with gradients (taken as it is) and without (transformed and kept)."""
    torch.manual_seed(0)
    layer = WinoConv2d(160, 64, 3, padding=1, device=dev, dtype=own)
    x = torch.randn(1, 160, 14, 14, device=dev, dtype=torch.float16).contiguous(memory_format=torch.channels_last)
    for step in range(4):
        with torch.no_grad():
            layer.weight.mul_(1.5)
            if step % 2:
                kept = layer(x)
        y = layer(x)
        w, b = layer.weight.detach().half(), layer.bias.detach().half()
        U = engine.transform_filter(w, x.shape, 1, 1, layer._tile_for(x.dtype), row=True)
        ref = engine.conv_forward(x, w, b, 1, 1, layer._tile_for(x.dtype), U=U, row=True)
        assert torch.equal(y.detach(), ref) and (not step % 2 or torch.equal(kept, ref))
        y.sum().backward()
        with torch.no_grad():
            layer.weight -= 1e-3 * layer.weight.grad
            assert torch.equal(layer(x), layer(x))


def _kept(layer):
    """The filter that the module's next pass finds, None if it finds none."""
    return layer._cache[1].on_stream() if layer._cache is not None and layer._cache[1].holds(layer.weight) else None


def _module(dev, own, seed):
    torch.manual_seed(seed)
    layer = WinoConv2d(160, 64, 3, padding=1, device=dev, dtype=own)
    x = torch.randn(1, 160, 14, 14, device=dev, dtype=torch.float16).contiguous(memory_format=torch.channels_last)
    assert _takes(x, layer.weight.detach().half()) == 1

    def reference(v):
        U = engine.transform_filter(layer.weight.detach().half(), v.shape, 1, 1, layer._tile_for(v.dtype), row=True)
        return engine.conv_forward(v.detach(), layer.weight.detach().half(), layer.bias.detach().half(), 1, 1, layer._tile_for(v.dtype), U=U, row=True)
    return layer, x, reference


@pytest.mark.skipif(not engine.USE_EXT, reason="no compiled host layer")
@pytest.mark.parametrize("own", [torch.float16, torch.float32])
@pytest.mark.parametrize("bias_too", [False, True])
def test_a_frozen_filter_is_kept_in_passes_with_gradients(dev, own, bias_too):
    """Where the input or the bias alone needs a gradient, the first pass makes the filter and the others find it."""
    layer, x, reference = _module(dev, own, 1)
    layer.weight.requires_grad_(False)
    layer.bias.requires_grad_(bias_too)
    x.requires_grad_(not bias_too)
    y = layer(x)
    U = _kept(layer)
    assert U is not None and y.requires_grad
    for _ in range(2):
        assert torch.equal(layer(x), y) and _kept(layer).data_ptr() == U.data_ptr()
    assert torch.equal(y.detach(), reference(x))
    with torch.no_grad():
        assert torch.equal(layer(x), y) and _kept(layer).data_ptr() == U.data_ptr()


@pytest.mark.skipif(not engine.USE_EXT, reason="no compiled host layer")
@pytest.mark.parametrize("own", [torch.float16, torch.float32])
def test_a_filter_is_kept_from_the_second_pass_on(dev, own):
    """A trained weight's first pass takes it as it is; the next with the same weight makes its filter, also on another batch size."""
    layer, x, reference = _module(dev, own, 2)
    more = torch.cat([x, -x]).contiguous(memory_format=torch.channels_last)
    for second in (x, more, x):
        y = layer(x)
        assert _kept(layer) is None and torch.equal(y.detach(), reference(x))
        y = layer(second)
        U = _kept(layer)
        assert U is not None and torch.equal(y.detach(), reference(second))
        assert torch.equal(layer(x).detach(), reference(x)) and _kept(layer).data_ptr() == U.data_ptr()
        y.sum().backward()
        with torch.no_grad():
            layer.weight -= 1e-3 * layer.weight.grad
