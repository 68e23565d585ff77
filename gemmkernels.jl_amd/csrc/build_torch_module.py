"""Builds the module between torch tensors and the library (gk_torch.cpp) for the torch and the interpreter that run this:

    python build_torch_module.py gk_torch.cpp gk_torch.so [--always]

It follows torch's ABI, so what it was built for is compiled in (``built_for`` of the package's _native.py, which loads no other) and it is built again where
that or the source has changed.  Where there is no torch for HIP, or no Python headers, it is left out: the library does not need it, and the package does without."""
import importlib.util
import os
import subprocess
import sys
import sysconfig


def main(source, out, always=False):
    def left_out(why):
        print(f"{os.path.basename(out)} is left out: {why}")
        return 0
    try:
        import torch
    except ImportError:
        return left_out(f"no torch for {sys.executable}")
    if torch.version.hip is None:
        return left_out("this torch is not one for HIP")
    headers = sysconfig.get_paths()["include"]
    if not os.path.exists(os.path.join(headers, "Python.h")):
        return left_out(f"no Python.h in {headers}")
    spec = importlib.util.spec_from_file_location("built_for", os.path.join(os.path.dirname(os.path.abspath(source)), "..", "gemmkernels", "_built_for.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    built_for = module.built_for()
    if not always and os.path.exists(out) and os.path.getmtime(out) >= max(os.path.getmtime(source), os.path.getmtime(__file__)):
        with open(out, "rb") as f:
            if built_for.encode() + b"\0" in f.read():
                return 0
    where = os.path.dirname(torch.__file__)
    os.makedirs(os.path.dirname(out), exist_ok=True)
    command = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
               f'-DGK_BUILT_FOR="{built_for}"', f"-I{where}/include", f"-I{where}/include/torch/csrc/api/include", f"-I{headers}", "-I/opt/rocm/include", source, "-o", out,
               f"-L{where}/lib", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    print(" ".join(command), flush=True)
    return subprocess.call(command)


if __name__ == "__main__":
    sys.exit(main(sys.argv[1], sys.argv[2], "--always" in sys.argv[3:]))
