"""The module between torch tensors and the library: loaded only by the interpreter and the torch that it was built for, and left out of the build without failing it where
there is no torch."""
import os
import subprocess
import sys

import pytest

from gemmkernels import _lib, _native

torch = pytest.importorskip("torch")
CSRC = os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "..", "csrc")


@pytest.fixture
def unloaded(monkeypatch):
    monkeypatch.setattr(_native, "_module", None)
    monkeypatch.setattr(_native, "_tried", False)


def test_it_loads_where_it_was_built(unloaded):
    assert _native.load() is not None and _native._built_for_of(_native._PATH) == _native.built_for()


def test_another_torch_does_not_load_it(unloaded, monkeypatch):
    monkeypatch.setattr(_native, "built_for", lambda: "cpython-310-x86_64-linux-gnu, torch 2.11.0 0")
    assert _native.load() is None


def test_a_module_that_does_not_say_is_not_loaded(unloaded, monkeypatch):
    monkeypatch.setattr(_native, "_PATH", _lib.LIB_PATH)                # (a library without gk_torch_built_for)
    assert _native.load() is None


def test_without_torch_the_build_leaves_it_out(tmp_path):
    out = tmp_path / "gk_torch.so"
    r = subprocess.run([sys.executable, "-S", os.path.join(CSRC, "build_torch_module.py"), os.path.join(CSRC, "gk_torch.cpp"), str(out)], capture_output=True, text=True)
    assert r.returncode == 0 and "no torch" in r.stdout and not out.exists(), r.stdout + r.stderr


def test_clean_takes_it_away():
    r = subprocess.run(["make", "-n", "-C", CSRC, "clean"], capture_output=True, text=True, check=True)
    assert "gk_torch.so" in r.stdout
