"""A transformed filter that a caller keeps (transform_filter "once per weight update"; the reference transforms it in every call:
src/split_kernel.cu:14-53) belongs to the layer, not to the batch or the image it was made for, wherever the plan's form is a
matter of the layer alone: every fp32 layer."""
import io
import itertools

import pytest
import torch

from pytorch_winoconv_amd import WinoConv2d, engine

IMAGES = [(1, 7, 7), (1, 14, 14), (2, 28, 28), (4, 14, 14), (16, 28, 28), (32, 28, 28), (3, 45, 61), (32, 56, 56)]


@pytest.mark.parametrize("m", [2, 4])
@pytest.mark.parametrize("kernel,stride", [((4, 4), 1), ((4, 5), 1), ((5, 5), 1), ((5, 4), 2), ((4, 4), 2), ((5, 5), 2), ((6, 6), 1), ((3, 3), 2), ((3, 3), 1), ((7, 7), 1)])
def test_form_of_fp32_layers_is_the_layers(m, kernel, stride):
    for C, K in itertools.product((3, 64, 160, 225, 256, 288, 512, 1024), (8, 64, 128, 256, 512)):
        forms = set()
        for n, h, w in IMAGES:
            d = engine.make_desc((n, C, h, w), (K, C) + kernel, torch.float32, stride, kernel[0] // 2, m, stacked=None, row=True)
            forms.add((d.stacked, d.direct, d.row, d.m))
        assert len(forms) == 1, (C, K, forms)


@pytest.mark.parametrize("kernel,C,K,apart", [
    ((5, 5), 224, 64, (0, 0)), ((5, 5), 225, 320, (1, 1)), ((5, 5), 256, 321, (1, 0)), ((5, 5), 257, 768, (1, 1)), ((5, 5), 512, 769, (1, 0)),
    ((4, 5), 224, 64, (0, 0)), ((4, 5), 225, 384, (1, 1)), ((5, 4), 512, 385, (1, 0)), ((4, 4), 512, 64, (0, 0)), ((6, 6), 512, 64, (0, 0)),
])
def test_where_the_pieces_of_fp32_layers_are_apart(kernel, C, K, apart):
    assert apart == tuple(int(engine.make_desc((2, C, 30, 30), (K, C) + kernel, torch.float32, 1, 2, m, stacked=None).stacked == 0) for m in (2, 4))


def test_filters_of_different_plans_differ_in_size():
    """The size is all that tells a filter of other options: the plan that is chosen has no other of its size in another order."""
    for kernel, stride, m, C, K in itertools.product(((4, 4), (4, 5), (5, 5), (3, 3)), (1, 2), (2, 4), (64, 256, 288, 512), (16, 512)):
        if kernel == (3, 3) and stride == 1:
            continue
        desc = lambda stacked: engine.make_desc((2, C, 30, 30), (K, C) + kernel, torch.float32, stride, 2, m, stacked=stacked, direct=False)
        size = lambda d: engine.plan_conv(d).t_total * engine._row(d, engine.plan_conv(d))
        if kernel == (4, 4):
            assert desc(None).stacked == 1        # both plans have four pieces of two taps an axis
        else:
            assert size(desc(False)) != size(desc(True))


@pytest.mark.gpu
@pytest.mark.parametrize("C,K,kernel,m,made,used", [
    (256, 256, (4, 4), 4, (16, 28, 28), (32, 28, 28)), (512, 512, (4, 4), 2, (1, 14, 14), (4, 14, 14)), (512, 512, (5, 5), 2, (4, 14, 14), (1, 14, 14)),
    (288, 512, (5, 5), 4, (1, 14, 14), (4, 28, 28)),
])
def test_filter_of_one_batch_in_another(dev, host_layer, C, K, kernel, m, made, used):
    g = torch.Generator().manual_seed(3)
    w = (torch.randn(K, C, *kernel, generator=g) * (2.0 / (C * kernel[0] * kernel[1])) ** 0.5).to(dev)
    x = torch.randn(used[0], C, *used[1:], generator=g).to(dev)
    U = engine.transform_filter(w, (made[0], C) + made[1:], 1, 2, m)
    assert torch.equal(engine.conv_forward(x, w, None, 1, 2, m, U=U), engine.conv_forward(x, w, None, 1, 2, m))


@pytest.mark.parametrize("kind", [engine.KeptFilter, engine._KeptFilter])
def test_the_weight_a_module_keeps_a_filter_of(kind):
    w = torch.nn.Parameter(torch.randn(8, 8, 3, 3), requires_grad=False)
    kept = kind(w, (0, 0, 4, 0, 2304))
    assert kept.holds(w) and kept.holds(w.detach()) and kept.holds(w.view(8, 8, 3, 3))
    assert not kept.holds(w.transpose(0, 1)) and not kept.holds(w.clone())
    w.add_(1)
    assert not kept.holds(w) and kind(w, (0, 0, 4, 0, 2304)).holds(w)
    place, kept = w.data_ptr(), kind(w, (0, 0, 4, 0, 2304))
    del w
    for _ in range(8):                           # another weight, perhaps where the first one was
        assert not kept.holds(torch.randn(8, 8, 3, 3))
    assert place


def test_modules_of_files_that_hold_a_filter():
    """Modules were once written with what they keep, a key and a tensor: what a pass would take for a filter of now."""
    layer = WinoConv2d(8, 16, 3, padding=1)
    state = dict(layer.__getstate__(), _cache=((0, 1, (9, 9), torch.float16, 4, (0, 0, 4, 0)), torch.zeros(36 * 16 * 32)), _plan=None)
    old = WinoConv2d.__new__(WinoConv2d)
    old.__setstate__(state)
    assert old._cache is None and old._plan is None and torch.equal(old.weight, layer.weight)
    file = io.BytesIO()
    torch.save(layer, file)
    file.seek(0)
    again = torch.load(file, weights_only=False)
    assert again._cache is None and torch.equal(again.weight, layer.weight) and again.padding == layer.padding
