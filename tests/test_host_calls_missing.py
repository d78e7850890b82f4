"""The native host calls are an addition: without them every call takes the general path."""
import subprocess
import sys

import pytest

import rumus_amd
from rumus_amd import _lib, ops


def test_without_the_native_host_calls(monkeypatch):
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.delattr(rumus_amd, "_host_calls", raising=False)
    monkeypatch.setitem(sys.modules, "rumus_amd._host_calls", None)       # an import of it fails
    with pytest.warns(RuntimeWarning, match="native host side"):
        assert ops._native("int8_linear", 1, 2, 3, None) is None
    assert ops._native("rumus_hip_qmatmul_int4", None) is None              # (and says so once)


def test_they_load_here():
    assert _lib.host().__name__ == "rumus_amd._host_calls"


def test_the_library_alone_builds_without_torch():
    plan = subprocess.run(["make", "-n", "-B", "-C", _lib.CSRC, "lib", "PYTHON=/nonexistent"], capture_output=True, text=True, check=True)
    assert "librumus_hip.so" in plan.stdout and "host_calls" not in plan.stdout and not plan.stderr
