"""The native call (csrc/host/mi_torch_call.cpp): it takes ordinary calls only, and answers as the Python body does."""

import numpy as np
import pytest
import torch

import kernel_library as kl
from kernel_library import _lib, _torch_call, config


def test_leaves_what_it_does_not_know_to_the_python_body():
    x = torch.zeros(8, 8, dtype=torch.bfloat16)
    assert _torch_call.call(0, x, x, None, 0.0, None) is None  # a CPU tensor
    assert _torch_call.call(0, None, x, None, 0.0, None) is None
    assert _torch_call.call(2, x, x, x, "eps", None) is None
    with pytest.raises(ValueError, match="HIP device"):
        kl.matmul_lhsT_rhs(x, x)
    with pytest.raises(TypeError):
        _torch_call.call(0, x, x)


def _mm(gpu, M=64, N=72, K=40, dtype=torch.bfloat16):
    g = torch.Generator(device=gpu).manual_seed(1)
    return (torch.randn(K, M, generator=g, device=gpu).to(dtype), torch.randn(K, N, generator=g, device=gpu).to(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["mm", "f32", "lhs", "rms", "online"])
def test_second_call_is_native_and_equal(gpu, kind):
    """The first call of a shape runs the Python body, the next ones the native call: the same bits, new or given output."""
    M, N, K = 64, 136, 88
    a, b = _mm(gpu, M, N, K, torch.float32 if kind == "f32" else torch.bfloat16)
    gamma = torch.linspace(0.5, 1.5, K, device=gpu).to(torch.bfloat16)
    if kind in ("mm", "f32"):
        def run(out=None): return kl.matmul_lhsT_rhs(a, b, out=out)
        def native(): return _torch_call.call(0, a, b, None, 0.0, None)
    elif kind == "lhs":
        a = a.t().contiguous()
        def run(out=None): return kl.matmul_lhs_rhs(a, b, out=out)
        def native(): return _torch_call.call(3, a, b, None, 0.0, None)
    else:
        a = a.t().contiguous()
        g = gamma if kind == "rms" else None
        def run(out=None): return kl.rmsnorm_matmul(a, b, g, eps=1e-5, out=out)
        def native(): return _torch_call.call(2, a, b, g, 1e-5, None)
    _torch_call.forget()
    assert native() is None
    first = run()
    second = native()
    assert second is not None and second.dtype == first.dtype and not second.requires_grad
    given = torch.full_like(first, float("nan"))
    assert run(out=given) is given
    assert torch.equal(first, second) and torch.equal(first, given)


@pytest.mark.gpu
def test_parameters_run_and_views_modes_and_transforms_do_not(gpu):
    a, b = _mm(gpu)
    want = kl.matmul_lhsT_rhs(a, b)
    p = torch.nn.Parameter(b)
    got = _torch_call.call(0, a, p, None, 0.0, None)
    assert torch.equal(got, want) and not got.requires_grad

    def native(x, y, out=None):
        return _torch_call.call(0, x, y, None, 0.0, out)

    class Sub(torch.Tensor):
        pass

    assert native(a.as_subclass(Sub), b) is None
    assert torch.equal(kl.matmul_lhsT_rhs(a.as_subclass(Sub), b), want)  # as the Python body always took it
    assert native(a, b.float()) is None and native(a, b.cpu()) is None
    assert native(a, b.t()) is None and native(a, b[:-8]) is None and native(a, b[:, :0]) is None
    assert native(a, b, out=b) is None and native(a, b, out=torch.empty(64, 64, device=gpu, dtype=a.dtype)) is None
    with pytest.raises(ValueError, match="contiguous"):
        kl.matmul_lhsT_rhs(a, b.t().contiguous().t())
    # An output that shares bytes with an input.
    store = torch.empty(40 * 64 + 64 * 72, device=gpu, dtype=a.dtype)
    x, out = store[: 40 * 64].view(40, 64), store[40 * 64 - 8 : 40 * 64 - 8 + 64 * 72].view(64, 72)
    assert native(x, b, out=out) is None
    with pytest.raises(ValueError, match="overlaps"):
        kl.matmul_lhsT_rhs(x, b, out=out)

    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    with TorchFunctionMode():
        assert native(a, b) is None
    with TorchDispatchMode():
        assert native(a, b) is None
    seen = []
    torch.func.vmap(lambda v: (seen.append(native(a, v)), v)[1])(b.expand(2, *b.shape))
    assert seen == [None]
    with torch.no_grad(), torch.autocast("cuda"):
        assert torch.equal(native(a, b), want)
    with torch.inference_mode():
        assert torch.equal(native(a, b), want)


@pytest.mark.gpu
def test_errors_of_the_library_are_raised(gpu):
    """A legality error of the C ABI comes back as the same exception as from the Python body."""
    a, b = _mm(gpu)
    kl.matmul_lhsT_rhs(a, b)
    shifted = torch.zeros(a.numel() + 1, device=gpu, dtype=a.dtype)[1:].view(a.shape)  # 2-byte aligned
    with pytest.raises(_lib.KernelLibraryError) as e:
        kl.matmul_lhsT_rhs(shifted, b)
    assert e.value.code == _lib.MI_E_ALIGN and "aligned" in str(e.value)
    r = kl.rmsnorm_matmul(a.t().contiguous(), b)
    with pytest.raises(_lib.KernelLibraryError) as e:
        kl.rmsnorm_matmul(a.t().contiguous(), b, eps=-1.0, out=r)
    assert e.value.code == _lib.MI_E_ARGS


@pytest.mark.gpu
def test_a_reloaded_tuned_table_is_followed(gpu):
    a, b = _mm(gpu)
    kl.matmul_lhsT_rhs(a, b)
    assert _torch_call.call(0, a, b, None, 0.0, None) is not None
    config.tuned_table(reload=True)
    assert _torch_call.call(0, a, b, None, 0.0, None) is None
    kl.matmul_lhsT_rhs(a, b)
    assert _torch_call.call(0, a, b, None, 0.0, None) is not None


@pytest.mark.gpu
def test_runs_on_the_current_stream(gpu):
    """Under capture on a side stream the call lands in the graph, which replays on new contents."""
    a, b = _mm(gpu)
    out = torch.empty(64, 72, device=gpu, dtype=a.dtype)
    kl.matmul_lhsT_rhs(a, b, out=out)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        kl.matmul_lhsT_rhs(a, b, out=out)
    for scale in (1.0, 2.0, -1.0):
        b.mul_(scale)
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.float().cpu().numpy(), kl.matmul_lhsT_rhs(a, b).float().cpu().numpy())
