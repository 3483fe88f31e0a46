"""Blocks 192 wide (three panels of 64), at the edges of the block, of K and of the rings.

Tolerance: a bf16 output is rounded once (2**-8 of its size between two
neighbours) and the fp32 sums differ from float64 by far less than 1e-2 of the
output's RMS over K products of random sign.  Each element is summed in the
same K order whatever the block, so an unsplit 192-wide block also gives the
very bits of a 128 x 128 one.
"""

import pytest

import kernel_library as kl

pytestmark = pytest.mark.gpu

LHST = ["bm192_bn256_bk32_w4_s3_v1", "bm192_bn192_bk32_w4_s3_v1", "bm192_bn128_bk32_w4_s3_v1", "bm128_bn192_bk32_w4_s3_v1"]
LHS = ["bm192_bn256_bk32_w8_s3_v1", "bm192_bn192_bk32_w4_s3_v1", "bm192_bn128_bk32_w4_s4_v1", "bm128_bn192_bk32_w4_s4_v1"]
# One block short of, of and past 64, 128 and 192; K of a part of a tile, of fewer tiles than the rings hold, odd and
# even numbers of tiles, and a tail.
SHAPES = [(8, 8, 8), (184, 200, 40), (192, 192, 96), (200, 184, 72), (264, 136, 328), (392, 584, 1032)]


def _inputs(M, N, K, device):
    import torch

    g = torch.Generator(device=device).manual_seed(M * 31 + N * 7 + K)
    x = torch.randn(M, K, generator=g, device=device).to(torch.bfloat16)
    return x, (torch.randn(K, N, generator=g, device=device) / K**0.5).to(torch.bfloat16)


def _check(out, exact):
    diff = (out.double() - exact).abs()
    floor = 1e-2 * float(exact.square().mean().sqrt())
    assert bool((diff <= floor + 1e-2 * exact.abs()).all()), float(diff.max())


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("name", LHST)
def test_lhst(gpu, name, M, N, K):
    x, w = _inputs(M, N, K, gpu)
    xt, exact = x.t().contiguous(), x.double() @ w.double()
    out = kl.matmul_lhsT_rhs(xt, w, cfg=kl.TileConfig.from_name(name))
    _check(out, exact)
    assert bool((out == kl.matmul_lhsT_rhs(xt, w, cfg=kl.TileConfig.from_name("bm128_bn128_bk32_w4_s4_v1"))).all())
    if K >= 328:
        _check(kl.matmul_lhsT_rhs(xt, w, cfg=kl.TileConfig.from_name(name + "_k3")), exact)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("name", LHS)
def test_lhs(gpu, name, M, N, K):
    x, w = _inputs(M, N, K, gpu)
    out = kl.matmul_lhs_rhs(x, w, cfg=kl.TileConfig.from_name(name))
    _check(out, x.double() @ w.double())
    assert bool((out == kl.matmul_lhs_rhs(x, w, cfg=kl.TileConfig.from_name("bm128_bn128_bk32_w4_s4_v1"))).all())


def test_only_the_cached_products_take_them():
    # The other variants refuse the block, as before.
    for func, variants in (("matmul_lhsT_rhs", (0, 2, 3, 4, 5, 6)), ("matmul_lhs_rhs", (0, 2)),
                           ("rmsnorm_matmul", (0, 1, 4, 5, 11, 12, 13, 14, 15, 16))):
        for v in variants:
            for block in ("bm192_bn128", "bm128_bn192"):
                code, _ = kl.check(func, kl.TileConfig.from_name(f"{block}_bk32_w4_s3" + (f"_v{v}" if v else "")), 1024, 1024, 1024)
                assert code != 0, (func, v, block)
