"""fp32 parameters rounded to the activations' type in one launch (layout_copy.hip): torch's values, where its threads and workgroups end."""
import pytest
import torch

from pytorch_winoconv_amd import WinoConv2d, _lib, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n_w,n_b", [(1, 0), (3, 1), (4, 5), (1023, 1024), (1025, 1027), (36864, 64)])
@pytest.mark.parametrize("start", [0, 1])
def test_torch_values(dev, dtype, n_w, n_b, start):
    g = torch.Generator().manual_seed(n_w)
    src = torch.randn(n_w + n_b + start, generator=g) * 10 ** torch.randint(-9, 6, (n_w + n_b + start,), generator=g).float()
    src[start] = float("inf")
    src = src.to(dev)
    w, b = src[start:start + n_w], src[start + n_w:]
    out = torch.full((n_w + n_b + start + 1,), 7.0, dtype=dtype, device=dev)
    wo, bo = out[start:start + n_w], out[start + n_w:start + n_w + n_b]
    _lib.check(_lib.load().wc_cast_parameters(engine._ptr(w), engine._ptr(wo), n_w, engine._ptr(b), engine._ptr(bo), n_b, engine._DTYPES[dtype], engine._stream(src)))
    assert torch.equal(wo, w.to(dtype)) and torch.equal(bo, b.to(dtype))
    assert float(out[-1]) == 7.0 and (start == 0 or float(out[0]) == 7.0)


@pytest.mark.parametrize("bias", [None, torch.float32, torch.float16])
@pytest.mark.parametrize("order", ["plain", "last", "wide"])
def test_modules_with_fp32_weights(dev, bias, order):
    torch.manual_seed(1)
    layer = WinoConv2d(64, 48, 3, padding=1, bias=bias is not None, device=dev)
    w = layer.weight.detach()
    if order == "last":
        w = w.contiguous(memory_format=torch.channels_last)
    if order == "wide":                        # not dense
        w = torch.cat([w, w], 1)[:, :64]
    layer.weight = torch.nn.Parameter(w)
    if bias is not None:
        layer.bias = torch.nn.Parameter(torch.randn(48, device=dev).to(bias))
    x = torch.randn(2, 64, 9, 9, device=dev, dtype=torch.float16).contiguous(memory_format=torch.channels_last).requires_grad_(True)
    y = layer(x)
    plain = WinoConv2d(64, 48, 3, padding=1, bias=bias is not None, device=dev, dtype=torch.float16)
    with torch.no_grad():
        plain.weight.copy_(layer.weight)
        if bias is not None:
            plain.bias.copy_(layer.bias)
    z = plain(x.detach())
    assert torch.equal(y.detach(), z.detach())
    y.sum().backward()
    assert layer.weight.grad.dtype == torch.float32 and layer.weight.grad.shape == layer.weight.shape
