"""fp32 layers of four pieces over many channels: the products of the pieces apart, on either side of the lines of the dispatch, against
fp64 (reference: the DWM plans of src/base_conv_launchers.h:58-388).  A tile of 4 amplifies fp32 rounding about tenfold: 2e-6 to 6e-6
in the 2-norm over these sums, stacked and apart."""
import pytest
import torch
import torch.nn.functional as F

import pytorch_winoconv_amd as pkg
from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 4])
@pytest.mark.parametrize("C,K,taps,stride,apart", [
    (224, 9, (5, 5), 1, False), (225, 9, (5, 5), 1, True), (256, 40, (4, 5), 1, True), (300, 33, (4, 4), 2, False), (270, 64, (5, 5), 2, True),
    (129, 20, (3, 3), 2, True), (320, 70, (3, 3), 2, True), (300, 16, (6, 6), 1, False), (300, 16, (3, 5), 1, False),
])
def test_against_fp64(dev, m, C, K, taps, stride, apart):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, C, 11, 14, generator=g)
    w = torch.randn(K, C, *taps, generator=g) * (2.0 / (C * taps[0] * taps[1])) ** 0.5
    b = torch.randn(K, generator=g)
    pad = (taps[0] // 2, taps[1] // 2)
    d = engine.make_desc(x.shape, w.shape, x.dtype, stride, pad, m, stacked=None)
    assert (d.stacked, d.direct) == (int(not apart), 0)
    want = F.conv2d(x.double(), w.double(), b.double(), stride, pad)
    got = engine.conv_forward(x.to(dev), w.to(dev), b.to(dev), stride, pad, m).cpu().double()
    assert (got - want).norm() <= 1e-5 * want.norm()


def test_module_with_changing_batches(dev):
    """The filter a module keeps is the plan's, and the gradients are those of the layer."""
    layer = pkg.WinoConv2d(288, 24, 5, padding=2, device=dev)
    for n in (1, 3, 3, 3, 1):
        x = torch.randn(n, 288, 9, 10, device=dev, requires_grad=True)
        y = layer(x)
        got = torch.autograd.grad(y.square().sum(), (x, layer.weight, layer.bias))
        x64, w64, b64 = (t.detach().cpu().double().requires_grad_(True) for t in (x, layer.weight, layer.bias))
        y64 = F.conv2d(x64, w64, b64, 1, 2)
        for a, e in zip((y,) + got, (y64,) + torch.autograd.grad(y64.square().sum(), (x64, w64, b64))):
            assert (a.cpu().double() - e).norm() <= 1e-5 * e.norm()
