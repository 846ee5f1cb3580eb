"""The row form on rows of x and y that are no multiple of 16 bytes, read and written as they lie: bit for bit what the same layer gives with
its channels padded with zeros (the reference pads to 32: src/base_conv_launchers.cu:325-352), infinities and NaN included, in every
shape of workgroup."""
import ctypes

import pytest
import torch

from pytorch_winoconv_amd import _lib, engine

pytestmark = pytest.mark.gpu

# N, C, K, spatial extents, taps; the last block of 32 channels holds 1 to 31 of them, the first one is the last one or not
CASES = [(1, 9, 24, (9, 11), 3), (1, 15, 33, (4, 5), 3), (2, 33, 35, (7, 13), 3), (1, 130, 66, (14, 14), 3), (1, 255, 40, (10, 9), 3), (2, 78, 17, (9, 8), 3),
         (1, 515, 39, (7, 7), 3), (3, 44, 200, (23, 30), 3), (1, 97, 130, (5, 61), 3), (1, 35, 9, (3, 2), 5), (2, 93, 41, (11, 12), 5), (1, 34, 45, (13, 10), 7),
         (1, 77, 32, (9, 20), 7), (1, 13, 40, (3, 6, 7), 3), (2, 70, 50, (4, 9, 9), 3), (1, 12, 7, (5, 6), 3), (1, 7, 32, (8, 9), 3), (1, 3, 36, (8, 9), 5)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_as_padded(dev, case, dtype, gemm_override):
    N, C, K, size, taps = case
    nd, pad, wide = len(size), taps // 2, (C + 7) // 8 * 8
    last = torch.channels_last if nd == 2 else torch.channels_last_3d
    g = torch.Generator().manual_seed(5)
    x = torch.randn(N, wide, *size, generator=g).to(dtype)
    w = (torch.randn(K, wide, *[taps] * nd, generator=g) * (2.0 / (C * taps ** nd)) ** 0.5).to(dtype)
    b = torch.randn(K, generator=g).to(dtype).to(dev)
    x[:, C:] = 0
    w[:, C:] = 0
    odd = x.clone()
    odd[0, C - 1].view(-1)[0] = float("inf")
    odd[-1, 0].view(-1)[-1] = float("nan")
    row = lambda c, k: engine.make_desc((N, c) + size, (k, c) + (taps,) * nd, dtype, 1, pad, 2, stacked=None, row=True).row
    if not row(C, K):
        pytest.skip("another form")
    K8 = (K + 7) // 8 * 8
    as_wide = row(wide, K8)              # the padded layer may have another form; channel-first x always comes through a padded copy
    w8, b8 = torch.zeros(K8, *w.shape[1:], dtype=dtype), torch.zeros(K8, dtype=dtype, device=dev)
    w8[:K], b8[:K] = w, b
    for config in [-1, 16, 18, 19] + ([17] if taps < 7 else []) + ([21] if taps == 3 else []):
        for t in (x, odd):
            ragged = t[:, :C].to(dev).contiguous(memory_format=last)
            gemm_override(config=config)
            got = engine.conv_forward(ragged, w[:, :C].to(dev), b, 1, pad, 2, row=True)
            first = engine.conv_forward(ragged.contiguous(), w[:, :C].to(dev), b, 1, pad, 2, row=True)
            gemm_override(config=config)
            want = engine.conv_forward(t.to(dev).contiguous(memory_format=last), w8.to(dev), b8, 1, pad, 2, row=True)[:, :K]
            if config >= 0 and as_wide:              # another shape may be chosen for another K
                assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
            assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), first.nan_to_num(7.0, 8.0, 9.0))


@pytest.mark.parametrize("C", [9, 20, 33])
def test_passes_of_a_batch(dev, C):
    x = torch.randn(5, C, 9, 10, device=dev).half().contiguous(memory_format=torch.channels_last)
    w = torch.randn(40, C, 3, 3, device=dev).half()
    whole = engine.conv_forward(x, w, None, 1, 1, 2, row=True)
    for chunk in (1, 2):
        assert torch.equal(engine.conv_forward(x, w, None, 1, 1, 2, chunk_images=chunk, row=True, channels_first_out=True), whole)
        assert torch.equal(engine.conv_forward(x.contiguous(), w, None, 1, 1, 2, chunk_images=chunk, row=True), whole)


@pytest.mark.parametrize("C,H", [(9, 9), (33, 9), (11, 7), (102, 45), (65, 9)])
def test_passes_that_start_anywhere(dev, host_layer, C, H):
    """Passes of a batch whose images of x are no multiple of 16 bytes: a channel-first y is written through a copy, x is read as it lies."""
    W = {45: 61, 7: 7}.get(H, 10)
    x = torch.randn(5, C, H, W, device=dev).half().contiguous(memory_format=torch.channels_last)
    w, b = torch.randn(40, C, 3, 3, device=dev).half(), torch.randn(40, device=dev).half()
    whole = engine.conv_forward(x, w, b, 1, 1, 2, row=True)
    for chunk in (1, 2, 3):
        assert torch.equal(engine.conv_forward(x, w, b, 1, 1, 2, chunk_images=chunk, row=True, channels_first_out=True), whole)
    # the entry points of the library: passes that it chooses itself, and an x that starts anywhere
    lib, y = _lib.load(), torch.empty(5, 40, H, W, device=dev, dtype=torch.float16)
    desc = engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 2, 1, stacked=None, row=True, y_layout=1)
    assert desc.row == 1
    _lib.check(lib.wc_conv_forward_static(ctypes.byref(desc), engine._ptr(x), engine._ptr(w), engine._w_strides(w), None, engine._ptr(b), engine._ptr(y), engine._stream(x)))
    assert torch.equal(y, whole)
    if C % 8:
        flat = torch.empty(x.numel() + 8, device=dev, dtype=torch.float16)
        view = flat[3:3 + x.numel()].copy_(x.permute(0, 2, 3, 1).reshape(-1))
        y.zero_()
        _lib.check(lib.wc_conv_forward_static(ctypes.byref(desc), engine._ptr(view), engine._ptr(w), engine._w_strides(w), None, engine._ptr(b), engine._ptr(y), engine._stream(x)))
        assert torch.equal(y, whole)


@pytest.mark.parametrize("C", list(range(1, 18)) + [31, 63, 100])
def test_padded_copy(dev, C, gemm_override):
    """The copy that tall boxes read, every remainder of the channel count."""
    x = torch.randn(1, C, 8, 9, device=dev).half().contiguous(memory_format=torch.channels_last)
    w = torch.randn(16, C, 3, 3, device=dev).half()
    if not engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 2, stacked=None, row=True).row:
        pytest.skip("another form")
    gemm_override(config=21)
    got = engine.conv_forward(x, w, None, 1, 1, 2, row=True)
    assert torch.equal(got, engine.conv_forward(x.contiguous(), w, None, 1, 1, 2, row=True))
    want = torch.nn.functional.conv2d(x.cpu().double(), w.cpu().double(), None, 1, 1)
    assert (got.cpu().double() - want).norm() <= 4e-3 * want.norm()       # U and V rounded to fp16: 5e-4 to 1e-3
