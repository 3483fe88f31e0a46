"""The second pass of split-K: every part count of its unrolled and general forms, both block sizes, both kernels.

Split and unsplit runs of one block add the same products in another
grouping, so each output of the split run is within two bf16 roundings
(2 * 2**-8 of its size) and the worst case of the fp32 regrouping
(K * 2**-23 of the sum of the products' magnitudes) of the unsplit one.
"""

import pytest

import kernel_library as kl

pytestmark = pytest.mark.gpu

# 48 x 232 outputs: blocks of 64 threads, the last one partly filled; 520 x 520: blocks of 256.
SHAPES = [(48, 232), (520, 520)]
PARTS = [2, 3, 4, 5, 8, 9, 16]


def _inputs(M, N, K, device):
    import torch

    g = torch.Generator(device=device).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=device).to(torch.bfloat16)
    w = (torch.randn(K, N, generator=g, device=device) / K**0.5).to(torch.bfloat16)
    return x, w, (1 + 0.1 * torch.randn(K, generator=g, device=device)).to(torch.bfloat16)


def _close(split, whole, magnitude, K):
    a, b = split.double(), whole.double()
    bound = 2 * 2.0**-8 * b.abs() + K * 2.0**-23 * magnitude + 1e-30
    assert bool(((a - b).abs() <= bound).all())


@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("parts", PARTS)
def test_matmul(gpu, M, N, parts):
    K = 64 * 79 + 40
    x, w, _ = _inputs(M, N, K, gpu)
    lhs_t = x.t().contiguous()
    cfg = kl.TileConfig(64, 64, 64, 4, 4, 1, 8, 1)
    whole = kl.matmul_lhsT_rhs(lhs_t, w, cfg=cfg)
    split = kl.matmul_lhsT_rhs(lhs_t, w, cfg=kl.TileConfig(64, 64, 64, 4, 4, parts, 8, 1))
    _close(split, whole, x.double().abs() @ w.double().abs(), K)


@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("parts", PARTS)
@pytest.mark.parametrize("variant", [4, 13])
def test_fused(gpu, M, N, parts, variant):
    """Variant 4 has as many row sums as parts, variant 13 one per 512 of K (10 here)."""
    K = 64 * 79 + 40
    x, w, g = _inputs(M, N, K, gpu)
    block = (128, 128, 64, 4, 2) if variant == 4 else (128, 128, 64, 4, 3)
    whole = kl.rmsnorm_matmul(x, w, g, cfg=kl.TileConfig(*block, 1, 8, variant))
    split = kl.rmsnorm_matmul(x, w, g, cfg=kl.TileConfig(*block, parts, 8, variant))
    scaled = x.double().abs() * g.double() * x.double().square().mean(1, keepdim=True).rsqrt()
    _close(split, whole, scaled @ w.double().abs(), K)
