"""The row form (wc_conv_desc.row; conv_row.hip): F(4,3) along the width axis, one kernel.  The reference has no such form
(its pieces are transformed along every axis: src/base_conv_launchers.cu:282-399); a convolution in fp64 pins it.

Bound: U and V are rounded once each, and with independent roundings of root mean square e the tile carries 3.1 e to the
output (points 0, +-0.652, +-1.534, infinity), whose own rounding adds e: in the 2-norm at most 4.1 e, e <= 2^-p / sqrt(3)
for p bits of significand (11 in fp16, 8 in bf16)."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import _lib, engine

pytestmark = pytest.mark.gpu
BOUND = {torch.float16: 4.1 * 2.0 ** -11 / 3 ** 0.5, torch.bfloat16: 4.1 * 2.0 ** -8 / 3 ** 0.5}

CASES = [
    # x shape, K, pad
    ((1, 32, 3, 3), 32, 1), ((2, 8, 1, 1), 1, 1),                      # one tile; one pixel
    ((2, 40, 13, 11), 33, 1),                                          # remainders of channels, blocks and tiles
    ((3, 33, 9, 17), 70, 0), ((1, 35, 6, 8), 129, (2, 0)),             # rows of x and of y that start anywhere
    ((5, 160, 7, 7), 100, 1), ((1, 264, 10, 5), 64, 1),                # channel blocks shared out unevenly
    ((9, 64, 14, 15), 136, 1), ((70, 32, 4, 4), 40, 1),                # boxes of several images, the last one short
    ((1, 72, 40, 65), 48, 1),
    ((2, 24, 5, 7, 9), 40, 1), ((1, 136, 3, 4, 6), 33, (1, 0, 1)), ((3, 40, 1, 9, 12), 64, 1), ((5, 32, 4, 5, 5), 32, (0, 1, 2)),
]


def _operands(xs, K, dtype, seed=1):
    g = torch.Generator().manual_seed(seed)
    nd = len(xs) - 2
    x = torch.randn(xs, generator=g).to(dtype)
    w = (torch.randn([K, xs[1]] + [3] * nd, generator=g) * (2.0 / (xs[1] * 3 ** nd)) ** 0.5).to(dtype)
    return x, w, torch.randn(K, generator=g).to(dtype)


def _err(y, ref):
    return float((y.double().cpu() - ref).norm() / ref.norm())


def _conv64(x, w, b, pad):
    conv = F.conv2d if x.dim() == 4 else F.conv3d
    return conv(x.double(), w.double(), None if b is None else b.double(), padding=pad)


def _row(x, w, b, pad):
    """The row form whatever the library would choose: through the C ABI."""
    lib = _lib.load()
    d = engine.make_desc(x.shape, w.shape, x.dtype, 1, pad, 2, x_layout=1)
    d.row = 1
    out, _ = engine.out_dims(d)
    n = ctypes.c_size_t()
    _lib.check(lib.wc_conv_workspace_bytes(ctypes.byref(d), ctypes.byref(n)))
    ws = torch.empty(n.value, dtype=torch.uint8, device=x.device)
    y = torch.full([x.shape[0]] + (out[1:] if x.dim() == 4 else out) + [w.shape[0]], float("nan"), dtype=x.dtype, device=x.device)
    _lib.check(lib.wc_conv_forward(ctypes.byref(d), x.data_ptr(), w.data_ptr(), engine._w_strides(w), None,
                                   b.data_ptr() if b is not None else None, y.data_ptr(), ws.data_ptr(), n.value,
                                   torch.cuda.current_stream().cuda_stream))
    return engine.channel_first_view(y)


@pytest.mark.parametrize("config", [16, 17, 18, 19])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_every_workgroup_shape_against_fp64(dev, dtype, case, config, gemm_override):
    xs, K, pad = case
    x, w, b = _operands(xs, K, dtype)
    gemm_override(config=config)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), _conv64(x, w, b, pad)) <= BOUND[dtype]
    assert _err(_row(x.to(dev), w.to(dev), None, pad), _conv64(x, w, None, pad)) <= BOUND[dtype]


def test_modules_and_layouts(dev, host_layer):
    """Where the library chooses the form: channel-first, channel-last and misaligned x and a cached filter give the same bits."""
    x, w, b = _operands((5, 256, 15, 14), 72, torch.float16)
    d = engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 4, stacked=None, row=True)
    assert d.row == 1 and engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 4, stacked=None).row == 0
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    y = engine.conv_forward(xd, wd, bd, 1, 1, 4, row=True)
    assert _err(y, _conv64(x, w, b, 1)) <= BOUND[x.dtype]
    xcl = xd.contiguous(memory_format=torch.channels_last)
    U = engine.transform_filter(wd, x.shape, 1, 1, 4, row=True)
    assert torch.equal(engine.conv_forward(xcl, wd, bd, 1, 1, 4, U=U, row=True), y)
    shifted = torch.empty(xd.numel() + 1, dtype=x.dtype, device=dev)[1:].view(5, 15, 14, 256).permute(0, 3, 1, 2)
    shifted.copy_(xd)
    assert torch.equal(engine.conv_forward(shifted, wd, bd, 1, 1, 4, U=U, row=True), y)
    assert torch.equal(engine.conv_forward(xd, wd, bd, 1, 1, 4, row=True, channels_first_out=True), y)
    mod = pkg.WinoConv2d(256, 72, 3, 1, 1, dtype=x.dtype, device=dev)
    with torch.no_grad():
        mod.weight.copy_(wd)
        mod.bias.copy_(bd)
        assert torch.equal(mod(xcl), y) and torch.equal(mod(xcl), y)
        mod.weight.mul_(2)
        assert _err(mod(xcl), _conv64(x, 2 * w, b, 1)) <= BOUND[x.dtype]


@pytest.mark.parametrize("dtype,ws,stride,m", [
    (torch.float32, (64, 64, 3, 3), 1, 2), (torch.bfloat16, (64, 64, 3, 3), 1, 2),       # one kernel where x is aligned
    (torch.float32, (40, 64, 3, 3), 1, 4), (torch.float16, (40, 64, 3, 3), 2, 2), (torch.float16, (40, 64, 5, 5), 1, 2),
])
def test_misaligned_operands_where_the_row_form_does_not_follow(dev, monkeypatch, dtype, ws, stride, m):
    """Permission for the row form copies nothing where the library takes another form, and both host layers run the same
    kernels: the same bits as without the permission."""
    g = torch.Generator().manual_seed(4)
    w = (torch.randn(ws, generator=g) * (2.0 / (ws[1] * ws[2] * ws[3])) ** 0.5).to(dtype).to(dev)
    x = torch.empty(2 * 64 * 15 * 14 + 1, dtype=dtype, device=dev)[1:].view(2, 15, 14, 64).permute(0, 3, 1, 2)
    x.copy_(torch.randn(x.shape, generator=g))
    assert engine.misaligned(x) and engine.make_desc(x.shape, ws, dtype, stride, ws[2] // 2, m, stacked=None, row=True).row == 0
    y = {}
    for compiled in (True, False):
        monkeypatch.setattr(engine, "USE_EXT", compiled)
        monkeypatch.setattr(torch.Tensor, "clone", lambda *_: pytest.fail("a copy"))
        y[compiled] = [engine.conv_forward(x, w, None, stride, ws[2] // 2, m, row=row) for row in (False, True)]
        monkeypatch.undo()
    assert all(torch.equal(v, y[True][0]) for v in y[True] + y[False])


@pytest.mark.parametrize("xs,K,chunk", [((5, 256, 7, 7), 64, 2), ((41, 156, 15, 14), 72, 7), ((3, 36, 4, 9, 10), 40, 1), ((70, 64, 30, 31), 130, 32)])
def test_passes_over_a_batch_give_the_bits_of_one_pass(dev, xs, K, chunk, host_layer):
    """Also where the whole batch and a pass would choose another shape of workgroup (shares of the channels or none)."""
    x, w, b = _operands(xs, K, torch.float16)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    d = engine.make_desc(xs, w.shape, x.dtype, 1, 1, 2, stacked=None, row=True)
    d.row = 1
    lib, fmt = _lib.load(), torch.channels_last if x.dim() == 4 else torch.channels_last_3d
    want = _row(xd, wd, bd, 1)
    assert _err(want, _conv64(x, w, b, 1)) <= BOUND[x.dtype]
    if engine.make_desc(xs, w.shape, x.dtype, 1, 1, 4, stacked=None, row=True).row:
        for x_in in (xd, xd.contiguous(memory_format=fmt)):
            for first in (False, True):
                y = engine.conv_forward(x_in, wd, bd, 1, 1, 4, chunk_images=chunk, row=True, channels_first_out=first)
                assert torch.equal(y, want)
    # the library's own scratch, in as many passes as fit
    for x_layout, x_in in ((1, xd), (0, engine.channel_last(xd))):
        d.x_layout, d.y_layout, d.chunk_images = x_layout, 1, chunk
        y = torch.full_like(want, float("nan")).contiguous()
        _lib.check(lib.wc_conv_forward_static(ctypes.byref(d), x_in.data_ptr(), wd.data_ptr(), engine._w_strides(wd), None, bd.data_ptr(),
                                              y.data_ptr(), torch.cuda.current_stream().cuda_stream))
        assert torch.equal(y, want)


def test_static_scratch_takes_a_batch_whose_copies_it_cannot_hold(dev):
    """132 MB of channel-first x in 64 MB of scratch."""
    x, w, b = _operands((41, 256, 80, 79), 32, torch.float16)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    d = engine.make_desc(x.shape, w.shape, x.dtype, 1, 1, 2, x_layout=1)
    d.row = 1
    y = torch.full((41, 80, 79, 32), float("nan"), dtype=x.dtype, device=dev)
    _lib.check(_lib.load().wc_conv_forward_static(ctypes.byref(d), xd.data_ptr(), wd.data_ptr(), engine._w_strides(wd), None,
                                                  bd.data_ptr(), y.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(engine.channel_first_view(y), _row(xd, wd, bd, 1))


def test_special_values_stay_in_their_windows(dev):
    """An infinity in x reaches the outputs whose tiles contain it and no others; padding channels never do."""
    x, w, _ = _operands((2, 36, 9, 24), 40, torch.float16)
    x[1, 35, 4, 9] = float("inf")
    y = _row(x.to(dev), w.to(dev), None, 1).cpu()
    assert bool(torch.isfinite(y[0]).all()) and not bool(torch.isfinite(y[1, :, 3:6, 8:11]).any())
    touched = torch.zeros(9, 24, dtype=torch.bool)
    touched[3:6, 4:12] = True                       # the tiles of four outputs whose six inputs hold column 9
    assert bool(torch.isfinite(y[1][:, ~touched]).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("xs,K,pad", [((70, 64, 30, 31), 136, 1), ((12, 40, 9, 30, 33), 40, 1), ((40, 72, 41, 29), 129, 0)])
def test_more_boxes_than_workgroups(dev, dtype, xs, K, pad, gemm_override):
    """Wide workgroups that go from box to box: boxes that do not share out evenly, the last of them partial."""
    x, w, b = _operands(xs, K, dtype)
    gemm_override(config=16)
    assert _err(_row(x.to(dev), w.to(dev), b.to(dev), pad), _conv64(x, w, b, pad)) <= BOUND[dtype]
