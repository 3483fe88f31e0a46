"""fp32 lhsT.rhs variant 3 (K split over the waves): every block and wave count at the edges of its tiles and chunks.

The reference is the float64 product; each output may differ from it by the
worst case of an fp32 sum of K products in any order, (K + 16) * 2**-23
times the sum of the products' magnitudes (16: the most waves whose sums
are added at the end; 2**-23 allows for truncated additions).
"""

import numpy as np
import pytest

import kernel_library as kl
from kernel_library import _lib

CONFIGS = [c.name for c in kl.compiled_configs("matmul_lhsT_rhs_f32") if c.variant == 3]

# (M, N, K): one element; one short of and past a 16-, 32- and 64-wide block; odd, even and 4-divisible rows (the
# loads' and stores' widths); K of less than a chunk, of a chunk short of a whole turn of the waves, and past one.
SHAPES = [(1, 1, 1), (15, 17, 33), (31, 33, 7), (63, 66, 127), (65, 62, 129), (64, 64, 512), (130, 68, 543),
          (33, 128, 1025)]


def _inputs(M, N, K, shift=0):
    import torch

    rng = np.random.default_rng(M * 7919 + N * 131 + K)
    host = [rng.standard_normal((K, c)).astype(np.float32) for c in (M, N)]
    dev = []
    for h in host:
        # `shift` floats into its storage: a 4-byte aligned operand.
        store = torch.zeros(h.size + shift, dtype=torch.float32, device="cuda:0")
        view = store[shift:].view(h.shape)
        view.copy_(torch.from_numpy(h))
        dev.append(view)
    return host, dev


def _check(out, a, b):
    K = a.shape[0]
    exact = a.astype(np.float64).T @ b.astype(np.float64)
    bound = (K + 16) * 2.0**-23 * (np.abs(a).astype(np.float64).T @ np.abs(b).astype(np.float64))
    err = np.abs(out.cpu().numpy().astype(np.float64) - exact)
    assert np.all(err <= bound), float((err - bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("name", CONFIGS)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_edges(gpu, name, M, N, K):
    (a, b), (da, db) = _inputs(M, N, K)
    _check(kl.matmul_lhsT_rhs(da, db, cfg=kl.TileConfig.from_name(name)), a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("name", CONFIGS)
def test_operands_aligned_to_four_bytes(gpu, name):
    """Even rows from an odd float offset: the 8-byte loads and 16-byte stores give way to narrow ones."""
    import torch

    M, N, K = 66, 68, 95
    (a, b), (da, db) = _inputs(M, N, K, shift=1)
    store = torch.full((M * N + 2,), 7.0, dtype=torch.float32, device="cuda:0")
    out = kl.matmul_lhsT_rhs(da, db, cfg=kl.TileConfig.from_name(name), out=store[1:-1].view(M, N))
    _check(out, a, b)
    assert store[0] == 7.0 and store[-1] == 7.0


@pytest.mark.gpu
@pytest.mark.parametrize("name", CONFIGS)
def test_nonfinite_operands_stay_in_their_rows_and_columns(gpu, name):
    """Columns past an edge read the neighbouring row: nothing of it may reach another output."""
    M, N, K = 37, 70, 67
    (a, b), (da, db) = _inputs(M, N, K)
    a[5, 0], a[66, 36], b[0, 69], b[40, 1] = np.inf, np.nan, -np.inf, np.inf
    for d, h in ((da, a), (db, b)):
        import torch

        d.copy_(torch.from_numpy(h))
    out = kl.matmul_lhsT_rhs(da, db, cfg=kl.TileConfig.from_name(name)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        exact = a.astype(np.float64).T @ b.astype(np.float64)
    assert np.array_equal(np.isfinite(out), np.isfinite(exact))
    assert np.array_equal(np.isnan(out), np.isnan(exact))
    inf = np.isinf(exact)
    assert np.array_equal(np.sign(out[inf]), np.sign(exact[inf]))


def test_default_is_the_split_kernel_wherever_its_offsets_reach():
    """Every shape whose operands stay under 4 GiB takes variant 3; a larger one keeps variant 1 and stays legal."""
    for M, N, K in [(1, 1, 1), (64, 64, 4096), (1000, 1501, 777), (4096, 4096, 4096), (7, 100003, 1), (32768, 64, 32767)]:
        c = kl.default_config("matmul_lhsT_rhs_f32", M, N, K)
        assert c.variant == 3 and kl.check("matmul_lhsT_rhs_f32", c, M, N, K)[0] == _lib.MI_OK
    for M, N, K in [(32768, 64, 32768), (64, 1 << 20, 1024), (1 << 25, 8, 1)]:
        c = kl.default_config("matmul_lhsT_rhs_f32", M, N, K)
        assert c.variant == 1 and kl.check("matmul_lhsT_rhs_f32", c, M, N, K)[0] == _lib.MI_OK
        rc, _ = kl.check("matmul_lhsT_rhs_f32", kl.TileConfig.from_name(CONFIGS[0]), M, N, K)
        assert rc == _lib.MI_E_RANGE
