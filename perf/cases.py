"""The calls that a program using kernel_library makes, as cases to be timed.

A case is one call of a public kernel at one shape:

* ``mm``      ``matmul_lhsT_rhs``, bf16 (lhs_T[K,M], rhs[K,N])
* ``f32``     ``matmul_lhsT_rhs``, fp32, any M, N and K
* ``lhs``     ``matmul_lhs_rhs``, bf16 (lhs[M,K], rhs[K,N])
* ``rms``     ``rmsnorm_matmul`` with gamma, bf16
* ``online``  ``rmsnorm_matmul_online`` (no gamma), bf16

``out`` says whether the caller brings the output buffer (a serving loop
that keeps its activations) or takes the one that the call allocates (the
online kernel always allocates).  No case passes a tile config: a program
takes the library's choice.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nki-autotune_amd"))

import kernel_library as kl  # noqa: E402

KINDS = ("mm", "f32", "lhs", "rms", "online")
MAX_FLOPS_BF16 = 2 * 8192**3
MAX_FLOPS_F32 = 2 * 4096**3
MAX_OPERAND = 28672 * 8192  # elements of the largest weight


def _case(name: str, kind: str, M: int, N: int, K: int, out: bool = False) -> dict:
    return {"name": name, "kind": kind, "M": M, "N": N, "K": K, "out": out}


def listed() -> list[dict]:
    return [
        # The smallest call a program makes: one block of work, so what counts is the call itself.
        _case("mm_small", "mm", 128, 192, 256),
        # The CPU-checkable fp32 product every kernel is compared with.
        _case("f32_small", "f32", 256, 512, 512),
        # fp32 at sizes that are no multiple of anything (fp32 takes any size).
        _case("f32_ragged", "f32", 1000, 1501, 777),
        # A large fp32 product, compute bound.
        _case("f32_large", "f32", 4096, 4096, 4096),
        # The reference kernel's own shape.
        _case("mm_2048", "mm", 2048, 2048, 2048),
        # The headline shape.
        _case("mm_8192", "mm", 8192, 8192, 8192),
        # A down projection over many rows: few output tiles, long K.
        _case("mm_down", "mm", 2048, 1024, 8192),
        # Decode of 16 rows against a large weight: bound by reading it.
        _case("mm_decode", "mm", 16, 28672, 8192, out=True),
        # Prefill of a ragged number of rows with row-major activations.
        _case("lhs_prefill", "lhs", 1000, 5000, 4104),
        # Norm and projection of a full block of rows.
        _case("rms_prefill", "rms", 4096, 4096, 4096),
        # Norm and projection of a few rows: latency bound.
        _case("rms_decode", "rms", 8, 4096, 4096, out=True),
        # The reference's fused kernel at its own shape, without gamma.
        _case("online_2048", "online", 2048, 2048, 2048),
    ]


def _spread(rng, lo: int, hi: int, step: int) -> int:
    """A multiple of ``step`` in [lo, hi], spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng) -> dict:
    kind = rng.choice(KINDS)
    while True:
        if kind == "f32":
            M, N, K = (_spread(rng, 64, 4096, rng.choice((1, 1, 8, 64))) for _ in range(3))
            limit = MAX_FLOPS_F32
        else:
            # A third of the calls are decode steps (8 to 128 rows), the others take a block of rows.
            rows = _spread(rng, 8, 128, 8) if rng.random() < 1 / 3 else _spread(rng, 128, 8192, 8)
            M, N, K = rows, _spread(rng, 128, 28672, 8), _spread(rng, 128, 16384, 8)
            limit = MAX_FLOPS_BF16
        if 2 * M * N * K <= limit and max(K * N, M * K, M * N) <= MAX_OPERAND:
            return {"kind": kind, "M": M, "N": N, "K": K, "out": kind != "online" and rng.random() < 0.5}


def _inputs(case: dict, seed: int) -> dict:
    """Inputs from the seed: U(-1,1) for the plain products (N(0, 0.02) weights and rows for a decode step),
    N(0,1) rows, gamma = 1 + 0.1 N(0,1) and N(0, 1/sqrt(K)) weights for the fused ones, N(0,1) in fp32."""
    kind, M, N, K = case["kind"], case["M"], case["N"], case["K"]
    dtype = torch.float32 if kind == "f32" else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)

    def uniform(*shape):
        return (torch.rand(shape, generator=g, device="cuda") * 2 - 1).to(dtype)

    if kind == "f32":
        return {"a": normal(K, M), "b": normal(K, N)}
    if kind in ("rms", "online"):
        d = {"a": normal(M, K), "b": normal(K, N, scale=1 / math.sqrt(K))}
        if kind == "rms":
            d["gamma"] = 1 + normal(K, scale=0.1)
        return d
    a_shape = (K, M) if kind == "mm" else (M, K)
    if M <= 128 and N >= 1024:
        return {"a": normal(*a_shape, scale=0.02), "b": normal(K, N, scale=0.02)}
    return {"a": uniform(*a_shape), "b": uniform(K, N)}


def prepare(case: dict, seed: int) -> dict:
    state = {"kind": case["kind"], **_inputs(case, seed), "out": None}
    if case["out"]:
        state["out"] = torch.empty((case["M"], case["N"]), dtype=state["a"].dtype, device="cuda")
    return state


def run(state: dict) -> torch.Tensor:
    kind = state["kind"]
    if kind in ("mm", "f32"):
        return kl.matmul_lhsT_rhs(state["a"], state["b"], out=state["out"])
    if kind == "lhs":
        return kl.matmul_lhs_rhs(state["a"], state["b"], out=state["out"])
    if kind == "rms":
        return kl.rmsnorm_matmul(state["a"], state["b"], state["gamma"], eps=kl.EPS, out=state["out"])
    return kl.rmsnorm_matmul_online(state["a"], state["b"])


def exact(case: dict, seed: int) -> torch.Tensor:
    """The same function of the same inputs in float64."""
    d = {k: v.double() for k, v in _inputs(case, seed).items()}
    if case["kind"] in ("mm", "f32"):
        return d["a"].t().contiguous() @ d["b"]
    if case["kind"] == "lhs":
        return d["a"] @ d["b"]
    x = d["a"]
    scale = torch.rsqrt(x.square().mean(dim=1, keepdim=True) + kl.EPS)
    return ((x * d["gamma"] if "gamma" in d else x) * scale) @ d["b"]


def work(case: dict) -> dict:
    M, N, K = case["M"], case["N"], case["K"]
    size = 4 if case["kind"] == "f32" else 2
    elements = M * K + K * N + M * N + (K if case["kind"] == "rms" else 0)
    return {"bytes": size * elements, "flops": 2 * M * N * K}


def tolerance(case: dict) -> dict:
    """Four times the distance from float64 that was measured over these ranges.

    bf16: 1.7e-3 (the rounding of the output) and 2.4e-3 with gamma (x * gamma is rounded to bf16 as well).
    fp32: 1.75e-8 times the root of K (the rounding of the running sum; 1.1e-6 at K = 4096).
    The largest single difference is about six times the relative error of a whole result."""
    if case["kind"] == "f32":
        rel = 7e-8 * math.sqrt(case["K"]) + 2e-7
    else:
        rel = 1e-2 if case["kind"] == "rms" else 7e-3
    return {"rel": rel, "max": 6 * rel}
