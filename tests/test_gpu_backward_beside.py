"""The weight gradient in the transform domain writes dw and, beside it, the bias gradient (backward.hip, backward_filter.hip): in one pass or by chunks of
images, through strides, in the operands' type or fp32."""
import ctypes

import pytest
import torch

from pytorch_winoconv_amd import _lib, engine

pytestmark = pytest.mark.gpu

CASES = [  # shape of x, output channels, taps, stride, tile
    ((3, 20, 9, 11), 24, 3, 1, 4), ((2, 33, 14, 14), 7, 5, 1, 2), ((4, 16, 8, 8), 40, 3, 2, 4), ((5, 8, 6, 5), 130, 7, 1, 2), ((2, 12, 4, 6, 7), 17, 3, 1, 2),
    ((3, 36, 4, 5, 6), 8, 3, 1, 4),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("xs,K,taps,stride,m", CASES)
def test_chunks_strides_and_types(dev, dtype, xs, K, taps, stride, m, gemm_override):
    gemm_override(config=20)                    # 16-bit 3x3 and 3x3x3 layers through the transform domain
    nd = len(xs) - 2
    g = torch.Generator().manual_seed(taps)
    out = [(s + 2 * (taps // 2) - taps) // stride + 1 for s in xs[2:]]
    x, dy = torch.randn(xs, generator=g).to(dtype), torch.randn([xs[0], K] + out, generator=g).to(dtype)
    shape = [K, xs[1]] + [taps] * nd
    conv = torch.nn.grad.conv2d_weight if nd == 2 else torch.nn.grad.conv3d_weight
    ref = conv(x.double(), shape, dy.double(), stride=stride, padding=taps // 2)
    ref_db = dy.double().sum([0] + list(range(2, nd + 2)))
    xd, dyd = engine.channel_last(x.to(dev)), engine.channel_last(dy.to(dev))
    lib = _lib.load()
    # fp32: the transforms' rounding, as in test_gpu_backward.py; 16 bits: V and dM are rounded to 11 bits and A^T of tile 4 grows that about tenfold
    bound = 1e-5 if dtype == torch.float32 else 2e-2
    seen = []
    for chunk in (0, 1, 2):
        for wide in (False, True):
            desc = engine.make_desc(xs, shape, dtype, stride, taps // 2, m, chunk, stacked=False)
            w_type = torch.float32 if wide else dtype
            # dw with its channels turned, as a view of a channels_last parameter's gradient
            dw = torch.empty([K] + [taps] * nd + [xs[1]], dtype=w_type, device=dev).permute([0, nd + 1] + list(range(1, nd + 1)))
            db = torch.empty(K, dtype=w_type, device=dev)
            n = ctypes.c_size_t()
            _lib.check(lib.wc_conv_backward_parameters_workspace_bytes(ctypes.byref(desc), ctypes.byref(n)))
            ws = torch.empty(n.value, dtype=torch.uint8, device=dev)
            _lib.check(lib.wc_conv_backward_parameters(ctypes.byref(desc), engine._ptr(xd), engine._ptr(dyd), engine._ptr(dw), engine._w_strides(dw),
                                                       engine._DTYPES[w_type], engine._ptr(db), engine._DTYPES[w_type], engine._ptr(ws), n.value, engine._stream(xd)))
            assert float((dw.double().cpu() - ref).abs().max() / ref.abs().max()) <= bound, (chunk, wide)
            # sums of at most a few hundred values in fp32, rounded to w_type
            assert float((db.double().cpu() - ref_db).abs().max() / ref_db.abs().max()) <= (1e-5 if wide or dtype == torch.float32 else 2e-3), (chunk, wide)
            seen.append(db.to(dtype))
    alone = engine.bias_gradient(dy.to(dev))
    assert all(torch.equal(s, alone) for s in seen)
