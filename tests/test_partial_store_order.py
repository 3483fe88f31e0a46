"""The split-K epilogue turns fragments between lanes through LDS: every turn from writes to reads and back to the next
fragment's writes is fenced, for both slot heights.

Without a fence the compiler, which sees only each thread's own addresses, may move a read above another lane's write
(or a later write above a read).  Read from the gfx950 assembly of a unit that holds the epilogue alone.  Needs hipcc,
not a GPU.
"""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

import build_lib

UNIT = """
#include "mi_gemm.hpp"
namespace mi {
#define MI_TEST_KERNEL(NAME, TM, TN, ROWS)                                                                         \\
  extern "C" __global__ __launch_bounds__(256) void NAME(const float* in, float* ws, int M, int N) {               \\
    __shared__ __attribute__((aligned(16))) char smem[4 * ROWS * kPartialRow];                                     \\
    f32x16_t acc[TM][TN];                                                                                          \\
    const int tid = (int)threadIdx.x;                                                                              \\
    for (int i = 0; i < TM; ++i)                                                                                   \\
      for (int j = 0; j < TN; ++j) acc[i][j] = ((const f32x16_t*)in)[(i * TN + j) * 256 + tid];                    \\
    store_partial<TM, TN, ROWS>(acc, ws, smem, tid >> 6, tid & 63, M, N, (int)blockIdx.x * TM * 32, 0);            \\
  }
MI_TEST_KERNEL(turns_2x2_32, 2, 2, 32)
MI_TEST_KERNEL(turns_1x2_16, 1, 2, 16)
}  // namespace mi
"""
KERNELS = ("turns_2x2_32", "turns_1x2_16")


def _unfenced(lines):
    """Pairs (write, read) and (read, write) of LDS accesses that some path runs with no wave barrier between them."""
    labels = {m.group(1): i for i, ln in enumerate(lines) if (m := re.match(r"^(\.LBB\w+):", ln))}
    bad = []
    for i, ln in enumerate(lines):
        m = re.match(r"\s*ds_(read|write)", ln)
        if not m:
            continue
        other = "ds_" + ("write" if m.group(1) == "read" else "read")
        seen, stack = set(), [i + 1]
        while stack:
            j = stack.pop()
            while j < len(lines) and j not in seen:
                seen.add(j)
                ins = lines[j].strip()
                if ins.startswith("; wave barrier") or ins.startswith("s_endpgm"):
                    break
                if ins.startswith(other):
                    bad.append((ln.strip(), ins))
                    break
                b = re.match(r"^s_(c?branch\w*)\s+(\.LBB\w+)", ins)
                if b:
                    stack.append(labels[b.group(2)])
                    if b.group(1) == "branch":
                        break
                j += 1
    return bad


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    tmp = tmp_path_factory.mktemp("turns")
    src, out = tmp / "turns.hip", tmp / "turns.s"
    src.write_text(UNIT)
    flags = [f for f in build_lib.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([hipcc, *flags, f"-I{build_lib.CSRC}", f"-I{build_lib.INCLUDE}", "--cuda-device-only", "-S", str(src),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


@pytest.mark.parametrize("name", KERNELS)
def test_every_turn_is_fenced(asm, name):
    body = asm.split(f"\n{name}:", 1)[1].split("\n.Lfunc_end", 1)[0]
    lines = body.split("\n")
    assert sum(ln.strip().startswith("ds_write") for ln in lines) and sum(ln.strip().startswith("ds_read") for ln in lines)
    bad = _unfenced(lines)
    assert not bad, bad[:3]
