"""The direct form of 16-bit types on LDS-DMA: every tile shape, forward and input gradient, against fp64.

Sizes at which it can go wrong: last tiles of pixels and channels that are partly or nearly empty, images that end inside a tile, taps
outside the image on every side, tiles over many small images, output rows past the image's end (wide padding), reductions shorter
than the loads in flight, kernels of one tap and of taps that a parity lacks."""

import pytest
import torch
import torch.nn.functional as F

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu

CASES = [
    # x shape, w shape, stride, pad
    ((1, 32, 4, 4), (8, 32, 1, 1), 2, 0), ((3, 32, 9, 5), (32, 32, 1, 1), 2, 0), ((2, 64, 17, 23), (72, 64, 3, 3), 2, 1), ((2, 160, 17, 23), (96, 160, 3, 3), 2, 1), ((3, 32, 16, 15), (136, 32, 3, 3), 2, 1),
    ((70, 32, 5, 3), (64, 32, 3, 3), 2, 1), ((2, 96, 9, 40), (264, 96, 2, 3), 2, (0, 1)), ((2, 32, 33, 31), (40, 32, 5, 5), 2, 2),
    ((5, 32, 6, 7), (32, 32, 3, 5), 2, (3, 5)), ((2, 32, 20, 18), (128, 32, 7, 7), 2, 3), ((2, 64, 12, 11), (64, 64, 5, 4), 1, (4, 3)),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [-1, 22, 23, 24, 25, 26])
@pytest.mark.parametrize("case", CASES)
def test_every_tile_is_exact_on_small_integers(dev, dtype, tile, case, gemm_override):
    """Integers whose sums stay below 2^24 in fp32, so that only the last rounding remains, the same on both sides."""
    xs, ws, stride, pad = case
    g = torch.Generator().manual_seed(3)
    x = torch.randint(-3, 4, xs, generator=g).double()
    w = torch.randint(-2, 3, ws, generator=g).double()
    b = torch.randint(-8, 9, (ws[0],), generator=g).double()
    want = F.conv2d(x, w, b, stride, pad)
    xd = x.to(dtype).to(dev).contiguous(memory_format=torch.channels_last)
    gemm_override(config=tile, rows_mode=0)
    y = engine.conv_forward(xd, w.to(dtype).to(dev), b.to(dtype).to(dev), stride, pad, 2, direct=True)
    assert torch.equal(y.cpu(), want.float().to(dtype))
    if stride == 2 and ws[0] % 32 == 0 and pad != (3, 5):       # other reductions are Winograd products, wider padding is refused
        dy = torch.randint(-3, 4, tuple(want.shape), generator=g).double()
        want = torch.nn.grad.conv2d_input(xs, w, dy, stride, pad)
        dx = engine.conv_backward_input(dy.to(dtype).to(dev).contiguous(memory_format=torch.channels_last), w.to(dtype).to(dev), xs[2:], stride, pad, 2)
        assert torch.equal(dx.cpu(), want.float().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_where_the_register_staged_kernel_takes_over(dev, dtype, gemm_override):
    """Forced here (kernel rows of more than 32 taps and images past 32-bit offsets take it by themselves)."""
    g = torch.Generator().manual_seed(4)
    x, w = torch.randint(-3, 4, (2, 32, 11, 13), generator=g).double(), torch.randint(-2, 3, (40, 32, 3, 3), generator=g).double()
    gemm_override(config=0)
    y = engine.conv_forward(x.to(dtype).to(dev), w.to(dtype).to(dev), None, 2, 1, 2, direct=True)
    assert torch.equal(y.cpu(), F.conv2d(x, w, None, 2, 1).float().to(dtype))
    dy = torch.randint(-3, 4, tuple(y.shape), generator=g).double()
    dx = engine.conv_backward_input(dy.to(dtype).to(dev), w.to(dtype).to(dev), (11, 13), 2, 1, 2)
    assert torch.equal(dx.cpu(), torch.nn.grad.conv2d_input((2, 32, 11, 13), w, dy, 2, 1).float().to(dtype))


@pytest.mark.parametrize("n,c,k,h,direct", [(1, 480, 64, 7, 1), (2, 384, 136, 9, 1), (1, 352, 32, 14, 1), (2, 384, 64, 9, 0)])
def test_reductions_that_left_the_parity_phases(dev, n, c, k, h, direct):
    """3x3 kernels at stride 2 over 356 to 500 channels, chosen by the library (but for fp32, the last): exact on small integers
    where no transform is taken."""
    dtype = torch.float16 if direct else torch.float32
    assert engine.make_desc((n, c, h, h), (k, c, 3, 3), dtype, 2, 1, 2, stacked=None).direct == direct
    g = torch.Generator().manual_seed(6)
    x, w = torch.randint(-3, 4, (n, c, h, h), generator=g).double(), torch.randint(-2, 3, (k, c, 3, 3), generator=g).double()
    y = engine.conv_forward(x.to(dtype).to(dev), w.to(dtype).to(dev), None, 2, 1, 2)
    want = F.conv2d(x, w, None, 2, 1)
    assert torch.equal(y.cpu(), want.float().to(dtype)) if direct else float((y.cpu() - want).abs().max()) <= 2e-4 * float(want.abs().max())


@pytest.mark.parametrize("shift", [1, 2, 4])
def test_tensors_that_start_anywhere(dev, shift):
    """x, dy and U that start 2, 4 or 8 bytes past a multiple of 16: through registers."""
    g = torch.Generator().manual_seed(8)
    x, w = torch.randint(-3, 4, (2, 64, 9, 11), generator=g).double(), torch.randint(-2, 3, (64, 64, 3, 3), generator=g).double()
    want = F.conv2d(x, w, None, 2, 1)
    dy = torch.randint(-3, 4, tuple(want.shape), generator=g).double()

    def moved(t):
        return torch.empty(t.numel() + 8, dtype=torch.float16, device=dev)[shift:shift + t.numel()].view(t.shape).copy_(t)

    def view(t):
        return moved(t.movedim(1, -1)).movedim(-1, 1)

    wd = w.half().to(dev)
    U = engine.transform_filter(wd, (2, 64, 9, 11), 2, 1, 2, direct=True)
    assert torch.equal(engine.conv_forward(view(x), wd, None, 2, 1, 2, U=U, direct=True).cpu(), want.half())
    assert torch.equal(engine.conv_forward(x.half().to(dev), wd, None, 2, 1, 2, U=moved(U), direct=True).cpu(), want.half())
    dx = engine.conv_backward_input(view(dy), wd, (9, 11), 2, 1, 2)
    assert torch.equal(dx.cpu(), torch.nn.grad.conv2d_input((2, 64, 9, 11), w, dy, 2, 1).half())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [-1, 1, 3, 4])
@pytest.mark.parametrize("case", [CASES[2], CASES[4], CASES[5], CASES[6], CASES[9], ((2, 64, 17, 40), (96, 64, 3, 3), 2, 1)])
def test_every_tile_through_registers(dev, dtype, tile, case, gemm_override):
    """Tensors that start two bytes past a multiple of 16, on the tile that their size asks for and on each of the three; the
    parity classes of an input gradient in one launch.  Exact on small integers."""
    xs, ws, stride, pad = case
    g = torch.Generator().manual_seed(9)
    x, w = torch.randint(-3, 4, xs, generator=g).double(), torch.randint(-2, 3, ws, generator=g).double()
    b = torch.randint(-8, 9, (ws[0],), generator=g).double()
    want = F.conv2d(x, w, b, stride, pad)

    def view(t):
        t = t.movedim(1, -1)
        return torch.full((t.numel() + 1,), float("nan"), dtype=dtype, device=dev)[1:].view(t.shape).copy_(t).movedim(-1, 1)

    wd = w.to(dtype).to(dev)
    U = engine.transform_filter(wd, xs, stride, pad, 2, direct=True)
    gemm_override(config=tile)
    assert torch.equal(engine.conv_forward(view(x), wd, b.to(dtype).to(dev), stride, pad, 2, U=U, direct=True).cpu(), want.float().to(dtype))
    if ws[0] % 32 == 0:
        dy = torch.randint(-3, 4, tuple(want.shape), generator=g).double()
        dx = engine.conv_backward_input(view(dy), wd, xs[2:], stride, pad, 2)
        assert torch.equal(dx.cpu(), torch.nn.grad.conv2d_input(xs, w, dy, stride, pad).float().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,c,k,h,w", [(8, 64, 32, 56, 56), (25, 128, 32, 31, 29), (7, 96, 64, 60, 1), (40, 32, 32, 33, 40)])
def test_classes_of_more_than_one_round_of_an_xcd(dev, dtype, n, c, k, h, w, gemm_override):
    """Input gradients whose launches have more workgroups than compute units, on the smallest tile: every tile of every class once, where
    an XCD's share is no multiple of the classes (8 x 784 pixels in tiles of 64: 49) and with two classes only.  Exact on small integers."""
    g = torch.Generator().manual_seed(11)
    wt = torch.randint(-2, 3, (k, c, 3, 3), generator=g).double()
    dy = torch.randint(-3, 4, (n, k, (h + 1) // 2, (w + 1) // 2), generator=g).double()
    if dtype == torch.float16:
        gemm_override(config=26)
    dx = engine.conv_backward_input(dy.to(dtype).to(dev).contiguous(memory_format=torch.channels_last), wt.to(dtype).to(dev), (h, w), 2, 1, 2)
    assert torch.equal(dx.cpu(), torch.nn.grad.conv2d_input((n, c, h, w), wt, dy, 2, 1).float().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [27, 28, 29])
@pytest.mark.parametrize("case", CASES + [((3, 96, 37, 41), (200, 96, 3, 3), 2, 1), ((2, 32, 30, 31), (128, 32, 1, 1), 1, 0), ((1, 32, 43, 42), (136, 32, 2, 1), 2, 0)])
def test_tall_tiles_are_exact_on_small_integers(dev, dtype, tile, case, gemm_override):
    """Forward products on tiles of 320, 384 and 448 pixels: odd and even counts of stages, fewer stages than the ring has places,
    last tiles of pixels and of channels that are nearly empty or of one row past a full one."""
    xs, ws, stride, pad = case
    g = torch.Generator().manual_seed(12)
    x = torch.randint(-3, 4, xs, generator=g).double()
    w = torch.randint(-2, 3, ws, generator=g).double()
    b = torch.randint(-8, 9, (ws[0],), generator=g).double()
    gemm_override(config=tile, rows_mode=0)
    y = engine.conv_forward(x.to(dtype).to(dev).contiguous(memory_format=torch.channels_last), w.to(dtype).to(dev), b.to(dtype).to(dev), stride, pad, 2, direct=True)
    assert torch.equal(y.cpu(), F.conv2d(x, w, b, stride, pad).float().to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("taps", [1, 2, 3])
def test_tall_tiles_pass_infinities_and_nan_on(dev, dtype, taps, gemm_override):
    """Odd and even counts of stages, the odd one with a stage of zeros behind it: what is no number reaches the pixels that read it, and no others."""
    g = torch.Generator().manual_seed(13)
    x = torch.randint(-3, 4, (2, 32, 41, 39), generator=g).double()
    x[0, 31, 40, 38], x[1, 0, 0, 0], x[1, 7, 20, 20] = float("inf"), float("nan"), float("-inf")
    w = torch.randint(1, 3, (136, 32, taps, taps), generator=g).double()
    w[5, 7] = float("inf")
    want = F.conv2d(x, w, None, 2).float().to(dtype)
    for tile in (27, 28, 29):
        gemm_override(config=tile, rows_mode=0)
        y = engine.conv_forward(x.to(dtype).to(dev).contiguous(memory_format=torch.channels_last), w.to(dtype).to(dev), None, 2, 0, 2, direct=True).cpu()
        assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(7.0), want.nan_to_num(7.0))
