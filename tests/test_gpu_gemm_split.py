"""fp32 wc_batched_gemm on the bf16 matrix cores (gemm.hip, Split): six of the nine products of three bf16 parts each.

Bound: what is left out is at most 2^-22 of a product; the sum is rounded (2^-24 of at most the sum of the absolute products)
six times per 16 channels, twice that allowed for what an instruction rounds inside."""
import pytest
import torch

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
