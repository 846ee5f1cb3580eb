"""wino_split / wino_concat of channel counts that are no multiple of a 16-byte vector, of tensors that start anywhere and of both memory
orders, bit for bit against the index maps of the oracle (reference: src/split_and_concat_kernels.cu:8-129)."""
import numpy as np
import pytest
import torch

from oracle import tiles as otiles
from pytorch_winoconv_amd import Split_and_Concat

pytestmark = pytest.mark.gpu


def _placed(t, shift, last, dev):
    """t on the GPU, `shift` elements into an allocation, channel-last or channel-first in memory"""
    order = [0] + list(range(2, t.dim())) + [1] if last else list(range(t.dim()))
    v = t.permute(order).contiguous()
    flat = torch.full((v.numel() + shift + 8,), 7, dtype=t.dtype, device=dev)
    view = flat[shift:shift + v.numel()].view(v.shape)
    view.copy_(v)
    return view.permute([order.index(i) for i in range(t.dim())])


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("shift", [0, 1, 6])
@pytest.mark.parametrize("last", [True, False])
@pytest.mark.parametrize("shape,wshape,m", [
    ((2, 119, 37, 41), (1, 119, 3, 3), 2), ((1, 70, 30, 19), (1, 70, 3, 3), 4), ((2, 65, 10, 63), (1, 65, 3, 3), 4), ((3, 7, 9, 8), (1, 7, 3, 3), 2),
    ((1, 1, 5, 6), (1, 1, 3, 3), 2), ((2, 72, 21, 150), (1, 72, 3, 3), 2), ((1, 33, 18, 138), (1, 33, 3, 3), 4), ((2, 15, 8, 12), (1, 15, 1, 1), 4),
    ((1, 9, 13, 11), (1, 9, 5, 5), 2), ((1, 19, 7, 9, 11), (1, 19, 3, 3, 3), 2), ((1, 66, 8, 7, 10), (1, 66, 3, 3, 3), 4), ((2, 10, 9, 8), (1, 10, 2, 2), 2),
])
def test_split(dev, dtype, shift, last, shape, wshape, m):
    x = torch.from_numpy(np.random.default_rng(1).integers(-999, 999, shape)).to(dtype)
    got = Split_and_Concat.wino_split(_placed(x, shift, last, dev), wshape, m)
    assert torch.equal(got.cpu(), torch.from_numpy(otiles.wino_split(x.numpy(), wshape, m)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("shift", [0, 1, 6])
@pytest.mark.parametrize("osize,K,B,m", [
    ((37, 41), 119, 2, 2), ((30, 19), 70, 1, 4), ((13, 63), 65, 1, 4), ((9, 8), 7, 2, 2), ((5, 6), 1, 1, 2), ((9, 11, 13), 19, 1, 2), ((8, 7, 10), 66, 1, 4),
    ((9, 10), 13, 2, 3),
])
def test_concat(dev, dtype, shift, osize, K, B, m):
    count = B * int(np.prod([-(-o // m) for o in osize]))
    t = torch.from_numpy(np.random.default_rng(2).integers(-999, 999, [count, K] + [m] * len(osize))).to(dtype)
    got = Split_and_Concat.wino_concat(_placed(t, shift, False, dev), osize, m)
    assert torch.equal(got.cpu(), torch.from_numpy(otiles.wino_concat(t.numpy(), osize, m)))


def test_strided_input_is_copied(dev):
    x = torch.randn(2, 12, 14, 9, device=dev).half()
    for v in (x[:, ::2], x[:, :, 1:], x.transpose(2, 3)):
        assert torch.equal(Split_and_Concat.wino_split(v, (1, v.shape[1], 3, 3), 2), Split_and_Concat.wino_split(v.contiguous(), (1, v.shape[1], 3, 3), 2))
