"""Another library through MI_KERNELS_LIB: its own picks, natively too, and none remembered from the one before."""

import shutil

import pytest

import kernel_library as kl
from kernel_library import _lib, _torch_call, config


@pytest.fixture
def other(tmp_path, monkeypatch):
    """A second library (a copy of the built one) and a switch to it."""
    path = shutil.copy(_lib.LIB_PATH, tmp_path / "libmi_other.so")
    return lambda: monkeypatch.setenv("MI_KERNELS_LIB", str(path))


def test_default_config_asks_the_library_in_use(other, monkeypatch):
    shape = (72, 200, 88)  # in no tuned table
    first = config.default_config("matmul_lhs_rhs", *shape)
    other()
    loaded = _lib.lib()
    asked = []

    class Spy:
        def __getattr__(self, name):
            asked.append(name)
            return getattr(loaded, name)

    monkeypatch.setattr(_lib, "lib", lambda: Spy())
    assert config.default_config("matmul_lhs_rhs", *shape) == first
    assert asked == ["mi_default_config"]
    config.default_config("matmul_lhs_rhs", *shape)
    assert asked == ["mi_default_config"]


@pytest.mark.gpu
def test_native_calls_follow_the_library(gpu, other):
    import torch

    _torch_call.forget()
    ops = [(torch.randn(40, 64, device=gpu).bfloat16(), torch.randn(40, n, device=gpu).bfloat16()) for n in (72, 80)]
    want = [kl.matmul_lhsT_rhs(a, b) for a, b in ops]

    def native(i):
        return _torch_call.call(0, *ops[i], None, 0.0, None)

    assert torch.equal(native(0), want[0]) and torch.equal(native(1), want[1])
    other()
    assert native(0) is None
    assert torch.equal(kl.matmul_lhsT_rhs(*ops[0]), want[0])
    # Bound to the other library now, which has seen the first shape only.
    assert torch.equal(native(0), want[0])
    assert native(1) is None
    assert torch.equal(kl.matmul_lhsT_rhs(*ops[1]), want[1]) and torch.equal(native(1), want[1])
    with pytest.raises(_lib.KernelLibraryError) as e:
        kl.rmsnorm_matmul(ops[0][0].t().contiguous(), ops[0][1], eps=-1.0)
    assert e.value.code == _lib.MI_E_ARGS
