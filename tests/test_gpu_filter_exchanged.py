"""The filter transform of filters whose output channels are closer in memory than their input channels (an input gradient's; the reference's
(kD, kH, kW, C, K) layout, dwm.py:85) against the same filter in torch's order, with gaps between its rows (a contiguous one has code of its own,
which rounds elsewhere), bit for bit."""
import pytest
import torch

from pytorch_winoconv_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,C", [(1, 5), (7, 32), (8, 33), (9, 64), (33, 100), (130, 40), (64, 260), (600, 256)])
@pytest.mark.parametrize("nd,m", [(2, 2), (2, 4), (3, 2)])
def test_exchanged(dev, dtype, K, C, nd, m):
    if nd == 3 and K * C > 20000:
        pytest.skip("as large as it needs to be")
    w = torch.randn(C, K, *[3] * nd, device=dev).to(dtype).transpose(0, 1)
    other = torch.randn(*[3] * nd, C, K, device=dev).to(dtype).permute(nd + 1, nd, *range(nd))
    shape = (2, C) + (12,) * nd
    for v in (w, other):
        a = engine.transform_filter(v, shape, 1, 1, m, stacked=False, direct=False)
        assert torch.equal(a, engine.transform_filter(torch.nn.functional.pad(v.contiguous(), (0, 1))[..., :3], shape, 1, 1, m, stacked=False, direct=False))
