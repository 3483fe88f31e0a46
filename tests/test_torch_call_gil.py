"""The native call reads nothing shared while it has given up the GIL: bind() and remember() write the library's entry
points and the shapes' configs under the GIL, on any thread that meets a new shape."""

import re
from pathlib import Path

import build_lib

SRC = Path(build_lib.CSRC) / "host" / "mi_torch_call.cpp"


def test_no_shared_state_without_the_gil():
    text = re.sub(r"//[^\n]*", "", SRC.read_text())
    shared = set(re.findall(r"\b(g_\w+)\b", text))
    assert {"g_lib", "g_configs"} <= shared
    regions = re.findall(r"Py_BEGIN_ALLOW_THREADS(.*?)Py_END_ALLOW_THREADS", text, re.S)
    assert regions
    for r in regions:
        assert not [g for g in shared if re.search(rf"\b{g}\b", r)], r
