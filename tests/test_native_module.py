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


@pytest.mark.parametrize("module", ["missing", "broken"])
def test_the_functions_need_the_library_alone(tmp_path, module):
    """a library made by its own target, or a torch that the module was not built for: calls go through ctypes"""
    package = tmp_path / "amdmigraphx_amd"
    package.mkdir()
    source = os.path.join(ROOT, "amdmigraphx_amd")
    for name in ("__init__.py", "capi.py", "ops.py", "lib"):
        os.symlink(os.path.join(source, name), package / name)
    if module == "broken":
        suffix = next(n for n in os.listdir(source) if n.startswith("_torch_calls.")).split(".", 1)[1]
        (package / f"_torch_calls.{suffix}").write_bytes(b"\x7fELF")
    got = _child("from amdmigraphx_amd import capi, ops; assert isinstance(ops._native, capi._NothingNative); "
                 "print(ops.quant_dot_workspace_size(16, 512, 8192) > 0)", cwd=tmp_path)
    assert got.returncode == 0, got.stderr
    assert got.stdout.split() == ["True"]
    assert ("cannot be loaded" in got.stderr) == (module == "broken")


def test_a_failed_build_shows_what_the_compiler_said(tmp_path, monkeypatch):
    (tmp_path / "csrc").mkdir()
    (tmp_path / "csrc" / "Makefile").write_text("all:\n\t@echo 'x.hip:7: error: no such builtin' >&2; exit 1\n")
    monkeypatch.setattr(capi, "_PKG", str(tmp_path))
    with pytest.raises(capi.Mi355Error, match="x.hip:7: error: no such builtin"):
        capi.build_library()


def test_a_call_that_is_not_plain_costs_next_to_nothing():
    """Outputs and workspaces of the caller's, other types and devices: these calls go on in Python, and are made by
    callers who allocate ahead to be fast.  (An exception for each took 2.3 us.)"""
    import time
    import torch
    native = capi.native()
    x, one = torch.ones(8, 8, dtype=torch.int8), torch.ones(1)
    calls = {"out": lambda: native.quant_dot(x, x, False, None, None, 0, 0, None, None, None, x, None, None),
             "device": lambda: native.quant_dot(x, x, False, None, None, 0, 0, None, None, None, None, None, None),
             "e5m2": lambda: native.quant_dot(x, x, "e5m2", None, None, 0, 0, None, None, None, None, None, None),
             "workspace": lambda: native.quant_convolution(x, x, None, None, None, 1, False, None, None, None, None, x),
             "scale": lambda: native.quantizelinear(x, one, None, 0)}
    for name, call in calls.items():
        assert call() is None
        best = 1.0
        for _ in range(50):
            start = time.perf_counter()
            for _ in range(100):
                call()
            best = min(best, (time.perf_counter() - start) / 100)
        assert best < 1e-6, (name, best)
