"""The row form of 5x5 and 7x7 kernels, F(2,5) and two of F(3,4) on the points of F(4,3) (conv_row.hip): the bound of
test_gpu_row.py, whose 3.1 e is at most 3.3 e here (the same points carry five taps to two outputs, four to three)."""
import pytest
import torch
import torch.nn.functional as F

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import dwm, engine
from test_gpu_row import _err, _row

pytestmark = pytest.mark.gpu
BOUND = {torch.float16: 4.3 * 2.0 ** -11 / 3 ** 0.5, torch.bfloat16: 4.3 * 2.0 ** -8 / 3 ** 0.5}

CASES = [
    ((2, 40, 5, 5), 33, 0), ((1, 32, 5, 6), 41, 2), ((2, 40, 13, 11), 33, 2),       # one pixel; a tile and a half; remainders
    ((3, 33, 9, 17), 70, (0, 4)), ((1, 35, 6, 8), 129, (4, 0)),                     # rows of x and of y that start anywhere
    ((5, 160, 7, 7), 100, 2), ((1, 264, 10, 5), 64, 1), ((9, 64, 14, 15), 136, 2), ((40, 32, 6, 6), 44, 2),
]


CASES_7 = [
    ((2, 40, 7, 7), 33, 0), ((1, 32, 7, 5), 41, 3), ((2, 40, 13, 11), 33, 3),       # one pixel; remainders of tiles and channels
    ((3, 33, 9, 17), 70, (0, 6)), ((1, 35, 6, 8), 129, (6, 0)), ((5, 160, 8, 7), 100, 3), ((9, 64, 14, 15), 136, 2),
    ((40, 32, 6, 6), 44, 3), ((1, 264, 10, 7), 40, 3),
]


def _operands(xs, K, dtype, seed=1, taps=5):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(xs, generator=g).to(dtype)
    w = (torch.randn([K, xs[1], taps, taps], generator=g) * (2.0 / (xs[1] * taps * taps)) ** 0.5).to(dtype)
    return x, w, torch.randn(K, generator=g).to(dtype)


@pytest.mark.parametrize("config", [16, 17, 18, 19])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("taps,case", [(5, c) for c in CASES] + [(7, c) for c in CASES_7])
def test_every_workgroup_shape_against_fp64(dev, dtype, taps, case, config, gemm_override):
    xs, K, pad = case
    x, w, b = _operands(xs, K, dtype, taps=taps)
    gemm_override(config=config)
    ref = F.conv2d(x.double(), w.double(), b.double(), padding=pad)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), ref) <= BOUND[dtype]


@pytest.mark.parametrize("taps", [5, 7])
def test_the_library_chooses_it(dev, host_layer, taps):
    """Channel-first, channel-last, cut into passes and with a cached filter: the same bits; a module's forward pass and input
    gradient; the functional interface; layers that keep the other plan."""
    x, w, b = _operands((3, 96, 21, 30), 72, torch.bfloat16, taps=taps)
    pad = taps // 2
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    ref = F.conv2d(x.double(), w.double(), b.double(), padding=pad)
    y = engine.conv_forward(xd, wd, bd, 1, pad, 2, row=True)
    assert _err(y, ref) <= BOUND[x.dtype] and engine.make_desc(x.shape, w.shape, x.dtype, 1, pad, 2, stacked=None, row=True).row == 1
    xcl = xd.contiguous(memory_format=torch.channels_last)
    U = engine.transform_filter(wd, x.shape, 1, pad, 2, row=True)
    assert torch.equal(engine.conv_forward(xcl, wd, bd, 1, pad, 2, U=U, row=True), y)
    assert torch.equal(engine.conv_forward(xd, wd, bd, 1, pad, 2, chunk_images=2, row=True), y)
    assert torch.equal(dwm.dwm2d(xcl, wd, bd, 1, pad, output_block=2), y)
    mod = pkg.WinoConv2d(96, 72, taps, 1, pad, dtype=x.dtype, device=dev)
    with torch.no_grad():
        mod.weight.copy_(wd)
        mod.bias.copy_(bd)
        assert torch.equal(mod(xcl), y)
    xg = xcl.requires_grad_(True)
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(2)).to(x.dtype)
    dx = torch.autograd.grad(mod(xg), xg, dy.to(dev))[0]
    xr = x.double().requires_grad_(True)
    want = torch.autograd.grad(F.conv2d(xr, w.double(), padding=pad), xr, dy.double())[0]
    assert _err(dx, want) <= BOUND[x.dtype]
    for K, dtype, row in ((40, torch.float16, 0), (41, torch.float16, 1), (33, torch.bfloat16, 0), (32, torch.bfloat16, 1), (64, torch.float32, 0)) if taps == 5 else ():
        for m in (2, 4):
            assert engine.make_desc((2, 64, 15, 14), (K, 64, 5, 5), dtype, 1, 2, m, stacked=None, row=True).row == row


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C", [256, 257, 288, 513])
def test_5x5_over_many_channels_keeps_the_more_exact_plan(dev, dtype, C):
    """Stacked pieces of F(2,3) and F(2,2), which tile 2 has above 256 channels, round less than F(2,5): 4.8e-3 | 5.2e-3 in bfloat16."""
    x, w, b = _operands((2, C, 20, 21), 96, dtype)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    ref = F.conv2d(x.double(), w.double(), b.double(), padding=2)
    row = engine.make_desc(x.shape, w.shape, dtype, 1, 2, 2, stacked=None, row=True).row
    assert row == (C <= 256) and engine.make_desc(x.shape, w.shape, dtype, 1, 2, 4, stacked=None, row=True).row == 1

    def err(y):
        return float((y.double().cpu() - ref).norm() / ref.norm())

    chosen = err(engine.conv_forward(xd, wd, bd, 1, 2, 2, row=True))
    assert chosen <= min(err(_row(xd, wd, bd, 2)), err(engine.conv_forward(xd, wd, bd, 1, 2, 2)))
