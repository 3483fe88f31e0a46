"""Default picks at shapes where a block was timed slower than another one that the rules offer: not the slower block.

Each entry: the shape, the slower block, and the times (us, calls back to back in interleaved rounds over three sets of
inputs, or over as many weights as no cache holds) of that block and of the faster one.
"""

import ctypes

import pytest

from kernel_library import _lib
from kernel_library.config import TileConfig

LHST, F32, FUSED, LHS, NO_GAMMA = range(5)

SLOWER = [
    # Without gamma: the gamma default's block, or its gamma-free form, behind the gamma-free choice of the rules.
    (NO_GAMMA, (264, 880, 122680), "bm64_bn64_bk64_w4_s4_v14", 821, 155),
    (NO_GAMMA, (208, 2264, 22400), "bm64_bn64_bk64_w4_s4_v14", 106, 58.7),
    (NO_GAMMA, (3808, 128, 2288), "bm64_bn128_bk64_w4_s4_v5_k4", 14.5, 10.3),
    (NO_GAMMA, (9824, 16, 5624), "bm256_bn128_bk32_w8_s3_v5_k4", 43.5, 31.7),
    (NO_GAMMA, (12936, 16, 8400), "bm256_bn128_bk32_w8_s3_v5_k4", 61.5, 48.0),
    (NO_GAMMA, (16928, 800, 1848), "bm256_bn128_bk32_w8_s3_v5", 87.0, 71.8),
    (NO_GAMMA, (60984, 208, 8), "bm256_bn128_bk32_w8_s3_v5", 10.6, 8.9),
    (NO_GAMMA, (3016, 7208, 168), "bm128_bn512_bk32_w8_s3_v4", 22.1, 20.6),
    (NO_GAMMA, (24, 5752, 320), "bm32_bn128_bk64_w4_s4_v5", 4.25, 3.98),
    (NO_GAMMA, (32, 44944, 80), "bm32_bn128_bk64_w4_s4_v5", 6.4, 5.05),
    (NO_GAMMA, (64, 37360, 16), "bm64_bn128_bk64_w4_s4_v5", 7.0, 5.4),
    # Three columns of tiles where one spans the output, with an x that no cache holds.
    (FUSED, (7168, 328, 14688), "bm256_bn128_bk32_w8_s3_v5_k3", 126.0, 110.1),
    (FUSED, (5368, 304, 8456), "bm256_bn128_bk32_w8_s3_v5_k4", 70.6, 62.6),
    (FUSED, (4464, 272, 10120), "bm256_bn128_bk32_w8_s3_v5_k4", 75.2, 66.9),
    (FUSED, (2664, 336, 15392), "bm128_bn128_bk32_w4_s4_v5_k4", 60.8, 56.6),
    (NO_GAMMA, (1536, 264, 50216), "bm256_bn128_bk32_w8_s3_v5_k12", 125.3, 90.5),
    (NO_GAMMA, (7032, 352, 13096), "bm256_bn128_bk32_w8_s3_v5_k3", 134.4, 101.4),
    # Short K, the output's stores its bound: smaller blocks.
    (LHST, (4072, 14904, 176), "bm256_bn128_bk32_w4_s3_v1", 59.3, 51.4),
    (LHST, (3496, 26040, 168), "bm256_bn128_bk32_w4_s3_v1", 85.9, 76.9),
    (LHST, (1224, 244688, 312), "bm128_bn256_bk32_w4_s3_v1", 407.0, 316.0),
    (LHST, (1240, 158800, 368), "bm256_bn128_bk32_w4_s3_v1", 267.0, 218.7),
    (LHS, (65344, 120, 344), "bm256_bn128_bk64_w8_s3", 15.2, 13.2),
    (LHS, (4832, 1648, 456), "bm256_bn128_bk64_w8_s3", 14.4, 13.5),
    (LHS, (400, 53104, 16), "bm128_bn128_bk32_w4_s4_v1", 15.1, 12.9),
    (LHS, (46328, 192, 8), "bm128_bn128_bk32_w4_s4_v1", 8.1, 7.4),
    # Skinny: one workgroup's chain over all of K.
    (LHST, (112, 752, 2288), "bm64_bn64_bk64_w4_s4_v1", 11.3, 8.6),
    (LHST, (120, 1248, 2128), "bm64_bn64_bk64_w4_s4_v1", 10.6, 8.8),
    (LHST, (128, 1352, 2312), "bm64_bn64_bk64_w4_s4_v1", 10.1, 9.1),
    (LHS, (80, 5928, 2224), "bm64_bn64_bk64_w4_s4_v2", 20.6, 17.3),
    (LHS, (104, 5384, 2456), "bm64_bn64_bk64_w4_s4_v2", 22.2, 18.9),
    # The same with the weight from HBM (800 MB of weights in turn).
    (LHST, (56, 1536, 1856), "bm64_bn64_bk64_w4_s4_v1", 12.4, 10.1),
    (LHST, (120, 1672, 1712), "bm64_bn64_bk64_w4_s4_v1", 15.0, 12.6),
    (LHST, (88, 376, 1608), "bm64_bn64_bk64_w4_s4_v1", 12.2, 10.4),
    (LHS, (56, 872, 1592), "bm64_bn64_bk64_w4_s4", 14.2, 10.1),
    (LHS, (8, 136, 1816), "bm64_bn64_bk64_w4_s4", 10.3, 8.0),
    (FUSED, (24, 3112, 1032), "bm32_bn128_bk64_w4_s4_v5", 11.9, 9.1),
    (NO_GAMMA, (64, 1584, 1112), "bm32_bn128_bk64_w4_s4_v5", 12.1, 9.1),
    (FUSED, (24, 744, 4312), "bm32_bn128_bk64_w4_s4_v5_k8", 11.4, 9.8),
    (FUSED, (16, 648, 5000), "bm32_bn128_bk64_w4_s4_v5_k16", 9.7, 8.9),
    (FUSED, (16, 9728, 232), "bm32_bn128_bk64_w4_s4_v5", 5.6, 5.3),
    (NO_GAMMA, (24, 480, 6776), "bm32_bn128_bk64_w4_s4_v5_k16", 10.8, 9.6),
]


def _default(kind, M, N, K):
    c = _lib.MiTileCfg()
    L = _lib.lib()
    rc = L.mi_default_config_no_gamma(M, N, K, ctypes.byref(c)) if kind == NO_GAMMA else \
        L.mi_default_config(kind, M, N, K, ctypes.byref(c))
    assert rc == _lib.MI_OK
    return TileConfig.from_c(c)


@pytest.mark.parametrize("kind,shape,slower,slow_us,fast_us", SLOWER)
def test_the_slower_block_is_not_picked(kind, shape, slower, slow_us, fast_us):
    assert fast_us < 0.96 * slow_us
    TileConfig.from_name(slower)
    assert _default(kind, *shape).name != slower
