"""The module of plain calls and the library beside it, from processes that have loaded nothing yet."""
import os
import subprocess
import sys

import pytest

from amdmigraphx_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(not os.path.exists(capi.lib_path()), reason="library not built in this checkout")


def _child(code, **kw):
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, **kw)


@pytest.mark.parametrize("first", ["", "capi.lib(); "])
def test_loads_where_torch_is_not(first):
    """as the build does: the module's libraries are torch's, which the process has not loaded"""
    got = _child("import sys; from amdmigraphx_amd import capi; assert 'torch' not in sys.modules; " + first +
                 "print(capi.native().__name__)", cwd=ROOT)
    assert got.returncode == 0, got.stderr
    assert got.stdout.split() == ["amdmigraphx_amd._torch_calls"]
