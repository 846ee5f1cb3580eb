"""fp32 products on the bf16 matrix cores (gemm.hip, Split), as whole layers take them where their error is the smaller one and
wc_batched_gemm on tiles forced here: six of the nine products of three bf16 parts each.

Bound: what is left out is at most 2^-22 of a product; the sum is rounded (2^-24 of at most the sum of the absolute products)
six times per 16 channels, twice that allowed for what an instruction rounds inside."""
import pytest
import torch
import torch.nn.functional as F

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu


def _check(M, V, U):
    ref = torch.bmm(V.double(), U.double().transpose(1, 2).contiguous())
    size = torch.bmm(V.double().abs(), U.double().abs().transpose(1, 2).contiguous())
    C = V.shape[2]
    assert bool(((M.double() - ref).abs() <= size * (2.0 ** -22 + 12 * C / 16 * 2.0 ** -24)).all())


@pytest.mark.parametrize("config", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("T,P,C,K", [(1, 1, 32, 8), (2, 63, 64, 72), (3, 129, 96, 136), (1, 257, 512, 64)])
def test_against_fp64_over_the_range_of_fp32(dev, T, P, C, K, config, gemm_override):
    g = torch.Generator().manual_seed(C + K)
    V, U = torch.randn(T, P, C, generator=g).to(dev), torch.randn(T, K, C, generator=g).to(dev)
    gemm_override(config=config)
    _check(engine.batched_gemm(V, U), V, U)
    V = V * 2.0 ** torch.randint(-60, 60, V.shape, generator=g).to(dev)
    U = U * 2.0 ** torch.randint(-40, 40, U.shape, generator=g).to(dev)
    _check(engine.batched_gemm(V, U), V, U)


def test_infinities_and_nan_stay_in_their_rows(dev):
    g = torch.Generator().manual_seed(3)
    V, U = torch.randn(2, 70, 64, generator=g).to(dev), torch.randn(2, 72, 64, generator=g).to(dev)
    M = engine.batched_gemm(V, U)
    top = torch.finfo(torch.float32).max
    for value in (float("inf"), -float("inf"), float("nan"), top):
        W = V.clone()
        W[1, 33, 17] = value
        got = engine.batched_gemm(W, U * 2.0 ** -8 if value == top else U)
        if value == top:
            assert bool(torch.isfinite(got).all())       # the largest number splits without overflow
            continue
        assert not bool(torch.isfinite(got[1, 33]).any())
        got[1, 33] = M[1, 33]
        assert torch.equal(got, M)


@pytest.mark.parametrize("config", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("value", [float("inf"), -float("inf")])
def test_an_infinity_keeps_its_sign(dev, value, config, gemm_override):
    """In either operand, against numbers with and without lower parts and against zero (no number then); every other sum
    keeps its bits."""
    g = torch.Generator().manual_seed(3)
    V, U = torch.randn(2, 150, 64, generator=g).to(dev), torch.randn(2, 136, 64, generator=g).to(dev)
    U[1, ::3, 17], U[1, 5, 17], V[0, ::3, 3], V[0, 149, 3] = -1.0, 0.0, 3.0, 0.0
    gemm_override(config=config)
    M = engine.batched_gemm(V, U)
    W = V.clone()
    W[1, 133, 17] = value
    got = engine.batched_gemm(W, U)
    assert torch.equal(torch.nan_to_num(got[1, 133], 7.0), torch.nan_to_num(value * U[1, :, 17], 7.0))
    got[1, 133] = M[1, 133]
    assert torch.equal(got, M)
    W = U.clone()
    W[0, 40, 3] = value
    got = engine.batched_gemm(V, W)
    assert torch.equal(torch.nan_to_num(got[0, :, 40], 7.0), torch.nan_to_num(value * V[0, :, 3], 7.0))
    got[0, :, 40] = M[0, :, 40]
    assert torch.equal(got, M)


@pytest.mark.parametrize("nd,C,K,stride", [(2, 20, 100, 1), (2, 20, 100, 2), (2, 64, 100, 1), (3, 20, 36, 1), (3, 32, 40, 1)])
def test_an_infinity_goes_through_layers_of_one_tap(dev, nd, C, K, stride):
    """A tile of one tap has nothing to transform: y, dx and dw are infinite where a plain sum is, with its sign."""
    g = torch.Generator().manual_seed(5)
    size = (9, 8, 7)[:nd]
    x, w = torch.randn(2, C, *size, generator=g), torch.randn(K, C, *[1] * nd, generator=g)
    x[(1, 7) + (4,) * nd], x[(0, 3) + (2,) * nd] = float("inf"), -float("inf")
    layer = (pkg.WinoConv2d if nd == 2 else pkg.WinoConv3d)(C, K, 1, stride=stride, bias=False, device=dev)
    with torch.no_grad():
        layer.weight.copy_(w)
    conv = F.conv2d if nd == 2 else F.conv3d

    def check(got, want):
        assert not bool(torch.isfinite(want).all())
        got, finite = got.detach().double().cpu(), torch.isfinite(want)
        assert torch.equal(got[~finite], want[~finite])
        if nd == 3 and got.shape[-1] > 1:       # outputs of a pair along the width meet in a product with zero
            finite = finite & finite[..., (torch.arange(got.shape[-1]) ^ 1).clamp(max=got.shape[-1] - 1)]
        assert bool(((got - want)[finite].abs() <= 1e-5 * want[finite].abs().max()).all())

    xd = x.to(dev).requires_grad_(True)
    y = layer(xd)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    yr = conv(xr, wr, stride=stride)
    check(y, yr.detach())
    dy = torch.randn(y.shape, generator=g)
    check(torch.autograd.grad(y, layer.weight, dy.to(dev))[0], torch.autograd.grad(yr, wr, dy.double(), retain_graph=True)[0])
    dy[(1, 11) + (1,) * nd] = float("inf")
    check(torch.autograd.grad(layer(xd), xd, dy.to(dev))[0], torch.autograd.grad(yr, xr, dy.double())[0])


LAYERS = [
    # kernel, stride, tile, channels: in parts from 64 to 1024 products a sum (512 for tiles of fewer than 36 elements), of transformed operands
    ((1, 1), 1, 4, 100), ((1, 1), 2, 2, 100), ((3, 3), 1, 2, 1), ((3, 3), 1, 4, 2), ((3, 3), 1, 2, 33), ((3, 3), 1, 4, 33), ((3, 3), 1, 2, 512), ((3, 3), 1, 4, 1024),
    ((3, 3), 1, 2, 2060), ((3, 3), 1, 4, 2060), ((1, 3), 1, 4, 256), ((4, 4), 1, 2, 520), ((5, 5), 1, 2, 128), ((5, 5), 1, 2, 512), ((5, 5), 1, 4, 256),
    ((5, 5), 1, 4, 512), ((7, 7), 1, 4, 64), ((2, 2), 2, 2, 64), ((3, 3), 2, 2, 256), ((3, 3), 2, 4, 132), ((3, 3), 2, 4, 512),
    ((3, 3, 3), 1, 2, 2), ((3, 3, 3), 1, 2, 64), ((1, 1, 1), 1, 2, 36), ((3, 3, 3), 2, 2, 8),
]


@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("ks,stride,m,C", LAYERS)
def test_no_larger_error_than_the_fp32_instructions(dev, ks, stride, m, C, kind, gemm_override):
    """Whole layers as the library takes them against the fp32 instructions, forced, both against fp64.  A twentieth for the spread of
    two errors over some ten thousand values."""
    nd = len(ks)
    g = torch.Generator(device=dev).manual_seed(C)
    x = torch.randn([2, C] + [14 if nd == 2 else 9] * nd, generator=g, device=dev)
    w = torch.randn([72, C, *ks], generator=g, device=dev) * (2.0 / (C * ks[0] * ks[-1])) ** 0.5
    x = x if kind == "normal" else x.relu() if kind == "relu" else x.abs()
    w = w.abs() if kind == "positive" else w
    ref = (F.conv2d if nd == 2 else F.conv3d)(x.double().cpu(), w.double().cpu(), stride=stride)

    def err():
        y = engine.conv_forward(x, w, None, stride, 0, m, unfused=True, direct=False)
        assert tuple(y.shape) == tuple(ref.shape)
        return float((y.double().cpu() - ref).norm() / ref.norm())

    chosen = err()
    gemm_override(config=22)
    assert chosen <= 1.05 * err()
