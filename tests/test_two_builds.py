"""Two builds of the library in one process do not call into each other."""
import os
import shutil
import subprocess
import sys

import pytest

from socu_amd._lib import LIB_PATH


def test_second_build_binds_its_own_functions(tmp_path):
    # Both are opened as the package opens its library (global scope).  The second
    # one's internal calls, whose argument structs may be laid out differently,
    # have to stay inside it: LD_DEBUG reports where each symbol was bound.
    if not os.path.exists(LIB_PATH):
        pytest.skip("library not built")
    first, second = tmp_path / "first.so", tmp_path / "second.so"
    shutil.copy(LIB_PATH, first)
    shutil.copy(LIB_PATH, second)
    code = f"import ctypes\nfor p in ({str(first)!r}, {str(second)!r}): ctypes.CDLL(p, mode=ctypes.RTLD_GLOBAL)"
    env = dict(os.environ, LD_DEBUG="bindings", LD_DEBUG_OUTPUT=str(tmp_path / "ld"), LD_BIND_NOW="1")
    subprocess.run([sys.executable, "-c", code], env=env, check=True, timeout=110)
    lines = [ln for f in tmp_path.glob("ld*") for ln in f.read_text(errors="replace").splitlines()]
    assert any(f"binding file {second} " in ln for ln in lines)
    crossed = [ln for ln in lines if f"binding file {second} " in ln and f" to {first} " in ln]
    assert not crossed, crossed[:5]
