"""The tap form of the weight gradient (backward_taps.hip; 16-bit 3x3 and 3x3x3 layers at stride 1).  The reference has no
backward pass (src/back/utils.cu:15-24); the gradient of a convolution in fp64 pins it.

Bound: the operands are exact and the sums fp32, so the result carries its own rounding, at most 2^-(p+1) of each value
relative for p + 1 bits of significand (11 in fp16, 8 in bf16), and the fp32 sum's: n 2^-24 of the sum of magnitudes for n
products, below 1e-5 of the 2-norm at these sizes."""
import pytest
import torch

from pytorch_winoconv_amd import _lib, engine

pytestmark = pytest.mark.gpu
BOUND = {torch.float16: 2.0 ** -11 + 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5}

CASES = [
    # x shape, K, pad
    ((1, 8, 3, 3), 8, 0),                                    # one output pixel
    ((1, 8, 1, 1), 8, 1),
    ((2, 8, 5, 6), 16, 1),
    ((3, 72, 9, 17), 136, 1),                                # remainders of channels on both sides, three blocks of 64
    ((1, 1, 1, 1), 1, 1), ((2, 7, 5, 6), 13, 1), ((3, 75, 9, 17), 133, 1), ((1, 3, 4, 3, 9), 5, 1),   # loads that cross the last channel
    ((2, 40, 7, 7), 72, 0), ((2, 64, 30, 50), 64, (2, 0)),   # other paddings
    ((1, 16, 4, 253), 24, 1), ((1, 16, 3, 254), 24, 1),      # the widest rows of the ring, and rows it does not hold
    ((5, 128, 31, 31), 256, 1),                              # several parts, the last one short
    ((1, 16, 4, 3, 9), 8, 1), ((2, 24, 3, 6, 5), 72, (0, 1, 2)), ((3, 64, 5, 12, 11), 128, 1),
]


def _last(t):
    return t.contiguous(memory_format=torch.channels_last if t.dim() == 4 else torch.channels_last_3d)


def _operands(xs, K, pad, dtype, seed=3):
    g = torch.Generator().manual_seed(seed)
    nd = len(xs) - 2
    pads = (pad,) * nd if isinstance(pad, int) else pad
    x = torch.randn(xs, generator=g).to(dtype)
    dy = torch.randn([xs[0], K] + [xs[2 + i] + 2 * pads[i] - 2 for i in range(nd)], generator=g).to(dtype)
    shape = (K, xs[1]) + (3,) * nd
    grad = torch.nn.grad.conv2d_weight if nd == 2 else torch.nn.grad.conv3d_weight
    return x, dy, pads, shape, grad(x.double(), shape, dy.double(), padding=pads)


def _err(dw, ref):
    return float((dw.double().cpu() - ref).norm() / ref.norm())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_against_fp64(dev, dtype, case):
    x, dy, pads, shape, ref = _operands(*case, dtype)
    dw = engine.conv_backward_weight(_last(x.to(dev)), _last(dy.to(dev)), shape, 1, pads, 2)
    wide = case[0][-1] == 254                                # the transform domain: test_gpu_backward.py's bound
    assert _err(dw, ref) <= (2e-2 if wide else BOUND[dtype])


@pytest.mark.parametrize("shift", [1, 4])
def test_tensors_that_start_anywhere(dev, shift):
    x, dy, pads, shape, ref = _operands((2, 24, 6, 7), 40, 1, torch.float16)

    def view(t):
        t = t.to(dev).permute(0, 2, 3, 1)
        flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=dev)[shift:shift + t.numel()]
        return flat.view(t.shape).copy_(t).permute(0, 3, 1, 2)

    dw = engine.conv_backward_weight(view(x), view(dy), shape, 1, pads, 2)
    assert _err(dw, ref) <= BOUND[torch.float16]


def test_parts_are_added_in_a_fixed_order(dev):
    x, dy, pads, shape, _ = _operands((5, 128, 31, 31), 256, 1, torch.float16)
    x, dy = _last(x.to(dev)), _last(dy.to(dev))
    first = engine.conv_backward_weight(x, dy, shape, 1, pads, 2)
    assert all(torch.equal(first, engine.conv_backward_weight(x, dy, shape, 1, pads, 2)) for _ in range(3))


def test_same_as_the_transform_domain(dev):
    """The tap form and the form it replaces agree within the second one's error."""
    x, dy, pads, shape, ref = _operands((3, 64, 5, 12, 11), 128, 1, torch.float16)
    x, dy = _last(x.to(dev)), _last(dy.to(dev))
    taps = engine.conv_backward_weight(x, dy, shape, 1, pads, 2)
    lib = _lib.load()
    _lib.check(lib.wc_test_gemm_override(20, 1))
    try:
        other = engine.conv_backward_weight(x, dy, shape, 1, pads, 2)
    finally:
        _lib.check(lib.wc_test_gemm_override(-1, 1))
    assert _err(taps, ref) < _err(other, ref)
    assert float((taps.float() - other.float()).norm() / taps.float().norm()) <= 5e-3


@pytest.mark.parametrize("n", [57343, 57344])
def test_positions_close_to_2g(dev, n):
    """The last images of a line of almost 2^31 positions: the largest that the tap form takes, and one that it leaves to the
    transform domain because the end of its last part would be 2^31.  Everything before the last two images is zero."""
    x = torch.zeros(n, 1, 169, 217, dtype=torch.bfloat16, device=dev)
    dy = torch.zeros_like(x)
    xl, dyl, pads, shape, ref = _operands((2, 1, 169, 217), 1, 1, torch.bfloat16)
    x[-2:], dy[-2:] = xl.to(dev), dyl.to(dev)
    # nine values of a sum over 73000 products: the transform domain as in test_gpu_backward.py
    assert _err(engine.conv_backward_weight(x, dy, shape, 1, pads, 2), ref) <= (BOUND[x.dtype] if n == 57343 else 2e-2)


DMA_CASES = [
    # x shape, K, pad: channels in multiples of 8, which LDS-DMA brings
    ((1, 8, 3, 3), 8, 0), ((1, 8, 1, 1), 8, (2, 1)), ((1, 8, 1, 1, 1), 8, 1),           # fewer steps than loads in flight
    ((2, 8, 9, 11), 72, 1), ((1, 64, 8, 16), 64, 1), ((3, 72, 20, 17), 136, (0, 2)),     # two steps and more; last channels on both sides
    ((70, 16, 1, 2), 24, 1), ((9, 16, 2, 1, 3), 136, (1, 2, 1)),                         # many small images and planes in a step
    ((1, 8, 4, 253), 24, 1), ((2, 136, 3, 6, 5), 200, (0, 1, 2)), ((4, 64, 33, 64), 64, 1),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", DMA_CASES)
def test_by_lds_dma_exact_on_small_integers(dev, dtype, case):
    """Integers whose sums stay below 2^24: exact in fp32, so only the last rounding remains, the same on both sides; NaN around x
    and dy in memory, which positions outside the image must not read."""
    xs, K, pad = case
    x, dy, pads, shape, _ = _operands(xs, K, pad, dtype)
    x, dy = (x * 2).round().clamp(-4, 4), (dy * 2).round().clamp(-4, 4)
    grad = torch.nn.grad.conv2d_weight if len(xs) == 4 else torch.nn.grad.conv3d_weight
    want = grad(x.double(), shape, dy.double(), padding=pads).float().to(dtype)

    def guarded(t):
        flat = torch.full((t.numel() + 4096,), float("nan"), dtype=dtype, device=dev)[2048:2048 + t.numel()]
        last = t.to(dev).movedim(1, -1)
        return flat.view(last.shape).copy_(last).movedim(-1, 1)

    assert torch.equal(engine.conv_backward_weight(guarded(x), guarded(dy), shape, 1, pads, 2).cpu(), want)
