"""Builds the host-compiled kernel headers of tests/native for CPU tests."""
import ctypes
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "hilbert_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def build(name, tmp_path_factory):
    """ctypes library of tests/native/<name>.cpp, compiled by the host compiler."""
    out = str(tmp_path_factory.mktemp("native") / (name + ".so"))
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-shared", "-fPIC", "-I", CSRC, "-I", os.path.join(ROCM, "include"),
                    os.path.join(HERE, "native", name + ".cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)
