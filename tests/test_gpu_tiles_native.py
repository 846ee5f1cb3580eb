"""wino_split and wino_concat through the compiled host layer: the bytes that the ctypes path gives for every memory order that either takes, the same
refusals, under capture and on another stream."""
import pytest
import torch

from pytorch_winoconv_amd import backend, engine, wino_concat, wino_split

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not engine.USE_EXT, reason="no compiled host layer")]


def _orders(x):
    last = torch.channels_last if x.dim() == 4 else torch.channels_last_3d
    wide = torch.empty(x.shape[:-1] + (x.shape[-1] + 3,), dtype=x.dtype, device=x.device)
    wide[..., :-3] = x
    return [x, x.contiguous(memory_format=last), wide[..., :-3], x.transpose(-1, -2).contiguous().transpose(-1, -2)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,taps,m", [((2, 8, 10, 14), 3, 2), ((1, 5, 9, 9), 3, 4), ((3, 33, 6, 6), 3, 4), ((2, 16, 11, 8), 5, 2), ((1, 3, 7, 9), 2, 3),
                                          ((2, 6, 4, 6, 8), 3, 2), ((1, 1, 4, 4), 3, 2)])
def test_as_through_ctypes(dev, monkeypatch, dtype, shape, taps, m):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(shape, generator=g).to(dtype).to(dev)
    w_shape = (7, shape[1]) + (taps,) * (len(shape) - 2)
    out = [s + 1 - taps for s in shape[2:]]
    per = 1
    for o in out:
        per *= -(-o // m)
    tiles = torch.randn((shape[0] * per, 7) + (m,) * len(out), generator=g).to(dtype).to(dev)

    def both():
        return ([wino_split(a, kind(w_shape), m) for a in _orders(x) for kind in (tuple, list, torch.Size)],
                [wino_concat(t, kind(out), m) for t in (tiles, tiles.transpose(0, 1).contiguous().transpose(0, 1)) for kind in (tuple, list)])

    native = both()
    assert engine._ext.wino_split(x, w_shape, m) is not None and engine._ext.wino_concat(tiles, out, m) is not None
    monkeypatch.setattr(engine, "USE_EXT", False)
    for a, b in zip(sum(native, []), sum(both(), [])):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def test_refused_as_before(dev):
    x = torch.randn(1, 4, 8, 8, device=dev)
    for args, error in [((x.cpu(), (4, 4, 3, 3), 2), ValueError), ((x.double(), (4, 4, 3, 3), 2), TypeError), ((x[0], (4, 4, 3, 3), 2), ValueError),
                        ((x, (4, 4, 3), 2), ValueError), ((x, (4, 4, 3, 3), 0), ZeroDivisionError)]:
        with pytest.raises(error):
            wino_split(*args)
    for args, error in [((x.cpu(), (8, 8), 2), ValueError), ((x, (8, 8, 8), 2), ValueError), ((torch.randn(3, 4, 2, 2, device=dev), (4, 4), 2), ValueError)]:
        with pytest.raises(error):
            wino_concat(*args)
    # extents whose product is a multiple of 2^64
    with pytest.raises(ValueError):
        wino_concat(torch.randn(1, 1, 1, 1, 1, device=dev), (1 << 22, 1 << 21, 1 << 21), 1)
    assert torch.equal(wino_split(x, (4, 4, 3.0, 3), 2), wino_split(x, (4, 4, 3, 3), 2))      # whatever int() takes


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("shape,size,m", [((16, 4, 2, 2), (16, 16), 4), ((16, 4, 4, 2), (16, 16), 4), ((16, 4, 4, 4), (8, 8), 2), ((16, 4, 1, 4), (8, 8), 2),
                                          ((8, 4, 2, 2, 2), (8, 8, 8), 4), ((8, 4, 3, 2, 2), (4, 4, 4), 2)])
def test_tiles_of_another_extent_are_refused(dev, monkeypatch, native, shape, size, m):
    """They would be read as tiles of m, beyond their memory where they are smaller."""
    monkeypatch.setattr(engine, "USE_EXT", native)
    tiles = torch.randn(shape, device=dev)
    with pytest.raises(ValueError):
        wino_concat(tiles, size, m)
    out = torch.empty((1,) + size + (4,), device=dev)
    concat = engine._ext.WinoConcat if native else backend.WinoConcat
    with pytest.raises(ValueError):
        concat(tiles, out, m, len(size) == 2)


def test_captured_and_on_another_stream(dev):
    x = torch.randn(2, 8, 10, 10, device=dev)
    tiles = torch.randn(2 * 16, 8, 2, 2, device=dev)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        there = wino_split(x, (8, 8, 3, 3), 2), wino_concat(tiles, (8, 8), 2)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kept = wino_split(x, (8, 8, 3, 3), 2), wino_concat(tiles, (8, 8), 2)
    for _ in range(3):
        x.normal_()
        tiles.normal_()
        graph.replay()
        assert torch.equal(kept[0], wino_split(x, (8, 8, 3, 3), 2)) and torch.equal(kept[1], wino_concat(tiles, (8, 8), 2))
    assert there[0].shape == kept[0].shape and there[1].shape == kept[1].shape
