"""The package imports in a tree that is not built, and beside an extension of another torch or Python; the build makes
that extension again."""

import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

import build_lib

CALLS = """
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import kernel_library as kl
    from autotune import search
print("warned:", [str(w.message) for w in seen if w.category is RuntimeWarning])
import torch
try:
    kl.matmul_lhsT_rhs(torch.zeros(8, 8), torch.zeros(8, 8))
except ValueError as e:
    print("refused:", e)
try:
    kl.default_config("matmul_lhsT_rhs", 264, 520, 88)
    print("picked")
except ImportError as e:
    print("not built:", e)
"""


def _run(tmp_path, *built):
    """CALLS in a copy of the package that holds the named built files only."""
    pkg = tmp_path / "pkg"
    shutil.copytree(build_lib.PKG_DIR, pkg, ignore=shutil.ignore_patterns("*.so", "_build", "__pycache__"))
    for name, content in built:
        if content is None:
            shutil.copy(build_lib.PKG_DIR / "kernel_library" / name, pkg / "kernel_library" / name)
        else:
            (pkg / "kernel_library" / name).write_bytes(content)
    env = {k: v for k, v in os.environ.items() if k != "MI_KERNELS_LIB"} | {"PYTHONPATH": str(pkg)}
    p = subprocess.run([sys.executable, "-c", CALLS], capture_output=True, text=True, env=env, cwd=tmp_path)
    assert p.returncode == 0, p.stderr[-2000:]
    return p.stdout


def test_an_unbuilt_tree_imports_and_names_the_build_command(tmp_path):
    out = _run(tmp_path)
    assert "warned: []" in out and "refused:" in out
    assert "not built:" in out and "build_lib.py" in out


def test_an_extension_that_does_not_load_leaves_the_python_body(tmp_path):
    out = _run(tmp_path, ("libmi_kernels.so", None), ("_torch_call.so", b"of another Python"))
    assert "build_lib.py" in out.split("warned:")[1].splitlines()[0]
    assert "refused:" in out and "picked" in out


def test_an_extension_of_another_torch_does_not_load(tmp_path):
    import torch

    data = (build_lib.PKG_DIR / "kernel_library" / "_torch_call.so").read_bytes()
    here = torch.__version__.split("+")[0].encode() + b"\0"
    assert here in data
    out = _run(tmp_path, ("libmi_kernels.so", None), ("_torch_call.so", data.replace(here, b"9" + here[1:])))
    assert "built for torch 9" in out.split("warned:")[1].splitlines()[0]
    assert "refused:" in out and "picked" in out


@pytest.mark.parametrize("stamp,builds", [(None, 1), ("torch 1.0, Python 3.0", 1), ("same", 0)])
def test_the_build_makes_the_extension_again_for_another_torch(tmp_path, monkeypatch, stamp, builds):
    lib = tmp_path / "_torch_call.so"
    lib.write_bytes(b"built")
    os.utime(lib, (2**33, 2**33))  # newer than its sources
    monkeypatch.setattr(build_lib, "TORCH_CALL", lib)
    monkeypatch.setattr(build_lib, "BUILD", tmp_path)
    ran = []

    def run(cmd, **_):
        ran.append(cmd)
        Path(cmd[cmd.index("-o") + 1]).write_bytes(b"built again")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(build_lib.subprocess, "run", run)
    if stamp == "same":
        build_lib._build_torch_call(True)
        os.utime(lib, (2**33, 2**33))
        ran.clear()
    elif stamp:
        (tmp_path / "torch_call.for").write_text(stamp)
    build_lib._build_torch_call(False)
    assert len(ran) == builds
