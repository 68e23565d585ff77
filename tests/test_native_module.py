"""The module between torch tensors and the library: left out of the build without failing it where
there is no torch."""
import os
import subprocess
import sys

from gemmkernels import _lib

CSRC = os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "..", "csrc")


def test_without_torch_the_build_leaves_it_out(tmp_path):
    out = tmp_path / "gk_torch.so"
    r = subprocess.run([sys.executable, "-S", os.path.join(CSRC, "build_torch_module.py"), os.path.join(CSRC, "gk_torch.cpp"), str(out)], capture_output=True, text=True)
    assert r.returncode == 0 and "no torch" in r.stdout and not out.exists(), r.stdout + r.stderr


def test_clean_takes_it_away():
    r = subprocess.run(["make", "-n", "-C", CSRC, "clean"], capture_output=True, text=True, check=True)
    assert "gk_torch.so" in r.stdout
