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


@pytest.fixture(params=["compiled", "ctypes", "python"])
def passes(request, monkeypatch):
    """Through the plan, past it, and without the compiled host layer's part of what is kept."""
    monkeypatch.setattr(engine, "USE_EXT", request.param == "compiled")
    if request.param == "python":
        monkeypatch.setattr(engine, "KeptFilter", engine._KeptFilter)
    return 4 if request.param == "compiled" else 1


_A_WHILE = 20_000_000                     # cycles: some ten milliseconds


@pytest.mark.parametrize("own", [torch.float16, torch.float32])
def test_a_filter_made_on_another_stream(dev, passes, own):
    """Two streams that are ordered behind the weight's update and not with each other: the one that comes second waits for the filter
    that the first one makes."""
    layer = pkg.WinoConv2d(64, 96, 5, padding=2, device=dev, dtype=own).requires_grad_(False)
    xa, xb = _input(dev, 2, 64, 15, 14), _input(dev, 2, 64, 15, 14, seed=2)
    for _ in range(passes):
        layer(xa)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for turn in range(3):
        layer.weight.mul_(-1.5)
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(_A_WHILE)
            ya = layer(xa)
        with torch.cuda.stream(b):
            yb = [layer(xb) for _ in range(2)]
        torch.cuda.synchronize()
        _close(ya, layer, xa)
        for y in yb:
            _close(y, layer, xb)


def test_a_filter_is_given_back_when_every_stream_is_through(dev, passes):
    """The filter is replaced, and its memory taken by others on the stream that it was made on, while another stream has yet to read it."""
    layer = pkg.WinoConv2d(64, 96, 5, padding=2, device=dev, dtype=torch.float16).requires_grad_(False)
    x = _input(dev, 2, 64, 15, 14)
    for _ in range(passes):
        layer(x)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    want = layer(x)
    with torch.cuda.stream(other):
        torch.cuda._sleep(_A_WHILE)
        got = layer(x)
    layer.weight.zero_()
    layer(x)                               # another filter; the first one's memory goes back
    U = engine.transform_filter(layer.weight, x.shape, 1, 2, 4, row=True)
    taken = [torch.full_like(U, 7.0) for _ in range(8)]
    torch.cuda.synchronize()
    assert torch.equal(got, want) and len(taken) == 8


@pytest.mark.parametrize("warm", [False, True])
def test_a_filter_made_inside_a_capture(dev, passes, warm):
    """It is there once the graph has been replayed and stays the graph's: passes outside make their own."""
    layer = pkg.WinoConv2d(64, 96, 5, padding=2, device=dev, dtype=torch.float16).requires_grad_(False)
    x = _input(dev, 2, 64, 15, 14)
    if warm:
        for _ in range(passes):
            layer(x)
        layer.weight.mul_(-1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = layer(x)
    taken = [torch.full((256, 1024), 7.0, device=dev) for _ in range(4)]
    eager = layer(x)
    _close(eager, layer, x)
    for i in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager) and torch.equal(layer(x), eager)
        x.copy_(_input(dev, 2, 64, 15, 14, seed=5 + i))
        eager = layer(x)
    assert len(taken) == 4


@pytest.mark.parametrize("own", [torch.float16, torch.float32])
@pytest.mark.parametrize("c,k,taps", [(64, 96, 5), (160, 64, 3)])
def test_a_captured_pass_of_a_trained_weight(dev, passes, own, c, k, taps):
    """Its graph is replayed after updates of the weight, whose filter the passes before the capture have kept, and gives what an eager pass does."""
    layer = pkg.WinoConv2d(c, k, taps, padding=taps // 2, device=dev, dtype=own)
    x = _input(dev, 2, c, 15, 14)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(max(passes, 3)):
            layer(x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = layer(x)
    assert y.requires_grad
    for i in range(3):
        with torch.no_grad():
            layer.weight.mul_(-1.5)
        x.copy_(_input(dev, 2, c, 15, 14, seed=5 + i))
        graph.replay()
        torch.cuda.synchronize()
        _close(y.detach(), layer, x)
        assert torch.equal(y, layer(x))


def test_a_filter_that_a_graph_reads_stays(dev, passes):
    """The module goes on with another type's and another weight's filter; the captured one's memory is not given to others."""
    layer = pkg.WinoConv2d(64, 96, 5, padding=2, device=dev).requires_grad_(False)
    x, other = _input(dev, 2, 64, 15, 14), _input(dev, 2, 64, 15, 14, dtype=torch.float32)
    for _ in range(passes):
        want = layer(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = layer(x)
    elems = engine.transform_filter(layer.weight.half(), x.shape, 1, 2, 4, row=True).numel()
    for change in (False, True):
        if change:
            layer.weight.mul_(-1)
        _close(layer(other), layer, other)
        _close(layer(x), layer, x)
        _close(layer(other), layer, other)
        taken = [torch.full((elems,), 7.0, dtype=torch.float16, device=dev) for _ in range(16)]
        for _ in range(2):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want) and len(taken) == 16


@pytest.mark.parametrize("own", [torch.float16, torch.float32])
def test_shapes_types_and_memory_orders_in_turn(dev, passes, own):
    """Each pass with the filter of its own form: batches on either side of the direct form's line, images, types and orders in memory."""
    layer = pkg.WinoConv2d(128, 128, 7, 2, 3, device=dev, dtype=own).requires_grad_(False)
    xs = [_input(dev, n, 128, h, w, dtype=t) for t in {torch.float16, own} for n, h, w in ((1, 30, 29), (40, 60, 60), (2, 31, 30))]
    forms = {engine.filter_form(x.shape, layer.weight.shape, x.dtype, 2, (3, 3), layer._tile_for(x.dtype))[0] for x in xs}
    assert forms == {0, 1}
    for turn in range(2):
        for x in xs + xs[::-1]:
            _close(layer(x), layer, x)
            _close(layer(x.contiguous()), layer, x)
        layer.weight.mul_(-1)


def test_images_of_one_plane_and_of_more_in_turn(dev, passes):
    """A kernel of one tap along the depth: the plan of a single plane has no tile along it, and a smaller filter."""
    layer = pkg.WinoConv3d(24, 16, (1, 3, 3), padding=(0, 1, 1), device=dev).requires_grad_(False)
    for turn in range(3):
        for depth in (1, 4, 1, 5):
            x = _input(dev, 2, 24, depth, 9, 10, dtype=torch.float32)
            want = F.conv3d(x.double(), layer.weight.double(), layer.bias.double(), 1, (0, 1, 1))
            assert (layer(x).double() - want).norm() <= 1e-5 * want.norm()
