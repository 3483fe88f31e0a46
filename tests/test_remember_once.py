"""A shape is handed to the native call once: calls that stay on the Python body (modes, subclasses) do not bind and
remember again each time."""

import pytest

from kernel_library import _lib, _torch_call, ops
from kernel_library.config import default_config


@pytest.fixture
def counted(monkeypatch):
    """ops with a counter of the shapes handed over."""
    calls = []

    class Counted:
        def __getattr__(self, name):
            return getattr(_torch_call, name)

        def remember(self, *a):
            calls.append(a[:4])
            return _torch_call.remember(*a)

    monkeypatch.setattr(ops, "_torch_call", Counted())
    _torch_call.forget()
    return calls


def test_once_per_shape_and_library(counted, monkeypatch, tmp_path):
    import shutil

    cfg = default_config("matmul_lhsT_rhs", 72, 88, 40)
    for _ in range(3):
        ops._remember(0, 72, 88, 40, cfg)
        ops._remember(3, 72, 88, 40, cfg)
    assert counted == [(0, 72, 88, 40), (3, 72, 88, 40)]
    assert _torch_call.knows(0, 72, 88, 40) and not _torch_call.knows(0, 72, 88, 48)
    monkeypatch.setenv("MI_KERNELS_LIB", str(shutil.copy(_lib.LIB_PATH, tmp_path / "libmi_other.so")))
    assert not _torch_call.knows(0, 72, 88, 40)
    ops._remember(0, 72, 88, 40, cfg)
    assert len(counted) == 3 and _torch_call.knows(0, 72, 88, 40)
    monkeypatch.delenv("MI_KERNELS_LIB")
    assert not _torch_call.knows(0, 72, 88, 40)
    ops._remember(0, 72, 88, 40, cfg)
    _torch_call.forget()
    ops._remember(0, 72, 88, 40, cfg)
    assert len(counted) == 5
    with pytest.raises(TypeError):
        _torch_call.knows(0, 1)


@pytest.mark.gpu
def test_calls_under_a_mode_hand_over_once(gpu, counted):
    import torch

    import kernel_library as kl

    a, b = torch.randn(40, 72, device=gpu).bfloat16(), torch.randn(40, 88, device=gpu).bfloat16()
    with torch.device(gpu):  # a mode: every call runs the Python body
        outs = [kl.matmul_lhsT_rhs(a, b) for _ in range(4)]
    assert counted == [(0, 72, 88, 40)]
    assert all(torch.equal(o, outs[0]) for o in outs) and torch.equal(kl.matmul_lhsT_rhs(a, b), outs[0])
    assert counted == [(0, 72, 88, 40)]
