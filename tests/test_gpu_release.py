"""``release_workspace`` has returned the memory when it returns: the device's free memory, which follows its frees about
1 ms later, is back each time (one look right after a release read the old figure in half of them)."""

import time

import pytest

import kernel_library as kl


@pytest.mark.gpu
def test_free_memory_is_back_after_each_release(gpu):
    import torch

    M = N = 8192
    K = 16384
    cfg = kl.TileConfig(256, 256, 32, 4, 3, split_k=4, variant=1)      # a workspace of 1 GiB
    a = torch.zeros((K, M), dtype=torch.bfloat16, device=gpu)
    b = torch.zeros((K, N), dtype=torch.bfloat16, device=gpu)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=gpu)
    kl.matmul_lhsT_rhs(a, b, cfg=cfg, out=out)
    torch.cuda.synchronize()
    kl.release_workspace()
    free = torch.cuda.mem_get_info(gpu)[0]
    for i in range(20):
        kl.matmul_lhsT_rhs(a, b, cfg=cfg, out=out)
        torch.cuda.synchronize()
        kl.release_workspace()
        held = free - torch.cuda.mem_get_info(gpu)[0]
        assert held <= 32 << 20, (i, held)
    # With nothing freed since, it waits for nothing.
    t = time.perf_counter()
    kl.release_workspace()
    assert time.perf_counter() - t < 3e-3
