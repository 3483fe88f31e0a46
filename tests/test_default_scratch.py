"""Default lhsT.rhs picks run from the no-allocation entry's static scratch: its contract is that a call without a
config never needs more (16 KiB of counters and split_k * M * N * 4 bytes)."""

import ctypes
import random

import pytest

from kernel_library import _lib

SCRATCH = 64 << 20
# 256 workgroups of 256 x 256: the partial products alone fill the scratch.
FULL = [(512, 8192, 12288), (1024, 4096, 16384), (1024, 8192, 12288), (2048, 2048, 12288), (4096, 2048, 12288),
        (8192, 512, 16384), (8192, 1024, 12288)]


def _bytes(M, N, K):
    c = _lib.MiTileCfg()
    assert _lib.lib().mi_default_config(0, M, N, K, ctypes.byref(c)) == _lib.MI_OK
    return c.split_k * M * N * 4 + 16384 if c.split_k > 1 else 0


@pytest.mark.parametrize("M,N,K", FULL)
def test_full_grids(M, N, K):
    assert _bytes(M, N, K) <= SCRATCH


def test_drawn_shapes():
    r = random.Random(0)
    shapes = [(128 * r.randint(1, 64), 128 * r.randint(1, 64), 256 * r.randint(1, 64)) for _ in range(20000)]
    shapes += [(8 * r.randint(1, 1024), 8 * r.randint(1, 2048), 8 * r.randint(1, 2048)) for _ in range(20000)]
    over = [s for s in shapes if _bytes(*s) > SCRATCH]
    assert not over, over[:5]
