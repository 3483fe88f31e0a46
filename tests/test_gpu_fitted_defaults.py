"""The blocks that the fitted default picks added, at the edges of their tiles, and default calls at drawn shapes.

Tolerance: a bf16 output is rounded once (2**-8 of its size between two
neighbours), x * gamma once more, and the fp32 sums differ by their order;
over K products of random sign that is far below 1e-2 of the output's RMS,
the floor that the oracle's own fused check uses.
"""

import random

import numpy as np
import pytest

import kernel_library as kl

pytestmark = pytest.mark.gpu

FUSED = ["bm128_bn128_bk32_w4_s4_v5", "bm64_bn128_bk64_w4_s4_v5", "bm64_bn64_bk64_w4_s4_v5", "bm32_bn128_bk64_w4_s4_v5",
         "bm32_bn128_bk64_w4_s4_v12"]
LHS = ["bm32_bn128_bk64_w4_s4_v2", "bm64_bn64_bk64_w4_s4_v2"]
# Rows and columns short of and past a block, K of a part of a tile, of fewer tiles than the rings hold, of whole turns
# of the rings (12 tiles of 64) and one past.
SHAPES = [(8, 8, 8), (40, 136, 72), (72, 120, 200), (136, 72, 768), (200, 264, 840)]


def _inputs(M, N, K, device):
    import torch

    g = torch.Generator(device=device).manual_seed(M * 31 + N * 7 + K)
    x = torch.randn(M, K, generator=g, device=device).to(torch.bfloat16)
    w = (torch.randn(K, N, generator=g, device=device) / K**0.5).to(torch.bfloat16)
    return x, w, (1 + 0.1 * torch.randn(K, generator=g, device=device)).to(torch.bfloat16)


def _fused(x, w, gamma):
    xd = x.double()
    y = xd * xd.square().mean(1, keepdim=True).add(1e-6).rsqrt()
    return (y if gamma is None else y * gamma.double()) @ w.double()


def _check(out, exact):
    diff = (out.double() - exact).abs()
    floor = 1e-2 * float(exact.square().mean().sqrt())
    assert bool((diff <= floor + 1e-2 * exact.abs()).all()), float(diff.max())


@pytest.mark.parametrize("name", FUSED)
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("parts", [1, 3])
def test_fused_blocks(gpu, name, M, N, K, parts):
    if parts > 1 and K < 768:
        parts = 1
    cfg = kl.TileConfig.from_name(name + (f"_k{parts}" if parts > 1 else ""))
    x, w, g = _inputs(M, N, K, gpu)
    for gamma in (g, None):
        _check(kl.rmsnorm_matmul(x, w, gamma, cfg=cfg), _fused(x, w, gamma))


@pytest.mark.parametrize("name", LHS)
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("parts", [1, 3])
def test_lhs_blocks(gpu, name, M, N, K, parts):
    if parts > 1 and K < 768:
        parts = 1
    x, w, _ = _inputs(M, N, K, gpu)
    _check(kl.matmul_lhs_rhs(x, w, cfg=kl.TileConfig.from_name(name + (f"_k{parts}" if parts > 1 else ""))),
           x.double() @ w.double())


@pytest.mark.parametrize("seed", range(24))
def test_default_calls(gpu, seed):
    """Default calls at shapes over the fitted range, each kind, against float64; twice, for the same bits."""
    rng = random.Random(seed)

    def size(lo, hi):
        return max(8, int(round(np.exp(rng.uniform(np.log(lo), np.log(hi))) / 8)) * 8)

    M, N, K = size(8, 128) if seed % 3 == 0 else size(129, 3000), size(64, 6000), size(64, 12000)
    print(M, N, K, flush=True)
    x, w, g = _inputs(M, N, K, gpu)
    for run, exact in ((lambda: kl.rmsnorm_matmul(x, w, g), _fused(x, w, g)),
                       (lambda: kl.rmsnorm_matmul_online(x, w), _fused(x, w, None)),
                       (lambda: kl.matmul_lhs_rhs(x, w), x.double() @ w.double()),
                       (lambda: kl.matmul_lhsT_rhs(x.t().contiguous(), w), x.double() @ w.double())):
        out = run()
        _check(out, exact)
        assert bool((out == run()).all())
