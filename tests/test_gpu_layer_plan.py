"""The modules' planned forward pass (LayerPlan of the compiled host layer) against the unplanned one, bit for bit.  The reference has no such modules that work (conv.py:324-339)."""
import copy
import threading

import pytest
import torch

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

LAYERS = [
    # module, x shape, out channels, kernel, stride, padding, bias, channel-first
    (pkg.WinoConv2d, (2, 40, 9, 11), 24, 3, 1, 1, True, False), (pkg.WinoConv2d, (2, 64, 15, 14), 64, 3, 1, 1, False, True),
    (pkg.WinoConv2d, (2, 16, 12, 13), 44, 5, 1, 2, True, True), (pkg.WinoConv2d, (2, 32, 15, 14), 32, 3, 2, 1, True, False),
    (pkg.WinoConv2d, (2, 3, 16, 16), 16, 7, 2, 3, True, False), (pkg.WinoConv2d, (1, 20, 1, 9), 12, 3, 1, 1, True, False),
    (pkg.WinoConv3d, (1, 24, 5, 6, 7), 40, 3, 1, 1, True, False), (pkg.WinoConv3d, (1, 16, 6, 7, 6), 16, 3, 2, 1, False, True),
]


def _layer(dev, case, dtype, own):
    kind, xs, K, taps, stride, pad, bias, first = case
    torch.manual_seed(4)
    layer = kind(xs[1], K, taps, stride=stride, padding=pad, bias=bias, device=dev, dtype=own)
    x = torch.randn(xs, device=dev).to(dtype)
    return layer, x if first else x.contiguous(memory_format=torch.channels_last if len(xs) == 4 else torch.channels_last_3d)


@pytest.mark.parametrize("dtype,own", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32), (torch.float16, torch.float64)])
@pytest.mark.parametrize("case", LAYERS)
def test_same_as_unplanned(dev, monkeypatch, case, dtype, own):
    layer, x = _layer(dev, case, dtype, own)
    if not layer._winograd_ok(x):
        pytest.skip("torch's own convolution")
    params = [layer.weight] + ([layer.bias] if case[6] else [])

    def step(planned):
        monkeypatch.setattr(engine, "USE_EXT", planned)
        with torch.no_grad():
            frozen = layer(x)
        t = x.clone(memory_format=torch.preserve_format).requires_grad_(True)
        y = layer(t)
        dy = torch.randn(y.shape, device=dev, generator=torch.Generator(dev).manual_seed(1)).to(dtype).contiguous(memory_format=torch.channels_last if y.dim() == 4 else torch.channels_last_3d)
        return (frozen, y) + torch.autograd.grad(y, [t] + params, dy)

    for _ in range(3):
        planned = step(True)
        for a, b in zip(planned, step(False)):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
        with torch.no_grad():                       # another weight, in place: U follows it
            layer.weight.mul_(0.5)
    assert layer._plan[1] is not None


def test_what_the_plan_leaves_to_python(dev):
    """Other shapes, strides, types, starts and hyperparameters; copies; a replaced weight."""
    layer, x = _layer(dev, LAYERS[0], torch.float16, torch.float16)
    layer.requires_grad_(False)
    for _ in range(3):
        y = layer(x)
    assert layer._plan[1] is not None
    other = copy.deepcopy(layer)
    assert other._plan is None and torch.equal(other(x), y)
    flat = torch.empty(x.numel() + 8, dtype=x.dtype, device=dev)
    for shift in (1, 4, 8):
        view = flat[shift:shift + x.numel()].view(2, 9, 11, 40).copy_(x.permute(0, 2, 3, 1)).permute(0, 3, 1, 2)
        assert torch.allclose(layer(view), y, atol=2e-2, rtol=2e-2)
    assert torch.equal(layer(x.contiguous()), y) and torch.equal(layer(x), y)
    assert torch.equal(layer(x[:1]), y[:1]) and torch.equal(layer(x[:, :, ::1, :]), y)
    layer.weight = torch.nn.Parameter(layer.weight * 2, requires_grad=False)
    layer.bias = None
    assert torch.allclose(layer(x), 2 * (y - other.bias.view(1, -1, 1, 1)), atol=2e-2, rtol=2e-2)
    layer.padding = (0, 0)
    assert layer(x).shape == (2, 24, 7, 9)
    with pytest.raises(ValueError):
        layer(x[:, :16])
    with pytest.raises(ValueError):
        layer(x.cpu())


def test_errors_of_the_backward_pass_keep_their_type(dev):
    layer = pkg.WinoConv2d(32, 32, 3, padding=3, device=dev)
    x = torch.randn(2, 32, 9, 9, device=dev, requires_grad=True)
    for _ in range(3):
        y = layer(x)
    with pytest.raises(NotImplementedError):
        y.sum().backward()


def test_threads_and_streams(dev):
    """One module in four threads, each on a stream of its own, weights frozen: a plan may be shared."""
    layer, x = _layer(dev, LAYERS[1], torch.float16, torch.float16)
    xs = [x + i for i in range(4)]
    with torch.no_grad():
        want = [layer(t) for t in xs]
    torch.cuda.synchronize()
    got = [None] * 4

    def work(i):
        with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got[i] = layer(xs[i])
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_weights_that_lie_where_the_last_one_did(dev):
    """New tensors in every call, freed after it; the same memory in another order; a module that was copied."""
    layer = pkg.WinoConv2d(24, 24, 3, padding=1, bias=False, device=dev, dtype=torch.float16).requires_grad_(False)
    x = torch.randn(2, 24, 10, 11, device=dev).half().contiguous(memory_format=torch.channels_last)
    places = set()
    for i in range(6):
        w = torch.full((24, 24, 3, 3), float(i), device=dev, dtype=torch.float16)
        places.add(w.data_ptr())
        y = torch.func.functional_call(layer, {"weight": w}, (x,))
        del w
        assert torch.equal(y, pkg.engine.conv_forward(x, torch.full((24, 24, 3, 3), float(i), device=dev, dtype=torch.float16), None, 1, 1, layer._tile_for(x.dtype), row=True))
    assert len(places) < 6
    w = torch.randn(24, 24, 3, 3, device=dev).half()
    for _ in range(2):
        for v in (w, w.transpose(0, 1), w.transpose(2, 3), w):
            y = torch.func.functional_call(layer, {"weight": v}, (x,))
            assert torch.equal(y, pkg.engine.conv_forward(x, v.contiguous(), None, 1, 1, layer._tile_for(x.dtype), row=True))
    assert copy.deepcopy(layer)._cache is None and torch.equal(copy.deepcopy(layer)(x), layer(x))
