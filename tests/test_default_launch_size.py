"""Default picks launch: fewer than 2**32 threads, wherever 64x64 blocks of 4 waves do (the largest outputs a GPU of
288 GB holds are near that)."""

import ctypes

import pytest

from kernel_library import _lib

# fp32 outputs of 69 to 270 GB over a short K, where small blocks are estimated fastest.
SHAPES = [(66000, 600000, 8), (60000, 600000, 8), (50000, 600000, 8), (8192, 1 << 22, 8), (1 << 18, 1 << 17, 4),
          (131072, 131072, 1), (200000, 200000, 8), (262143, 250000, 2), (64, 1 << 25, 1)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp32(M, N, K):
    c = _lib.MiTileCfg()
    assert _lib.lib().mi_default_config(1, M, N, K, ctypes.byref(c)) == _lib.MI_OK
    assert _lib.lib().mi_cfg_check(1, ctypes.byref(c), M, N, K) == _lib.MI_OK
    tiles = -(-M // c.block_m) * -(-N // c.block_n)
    assert -(-M // 64) * -(-N // 64) * 256 < 2**32
    assert tiles * c.waves * 64 < 2**32
