"""Calls the host functions of csrc/route.h through a small shared library."""
import ctypes
import os
import subprocess

from saclaymocks_amd import _lib

CSRC = os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "csrc")


def build(tmp_path, declarations):
    """A library of `declarations`, C++ definitions that use smk_route's functions."""
    src, lib = str(tmp_path / "rules.cpp"), str(tmp_path / "rules.so")
    with open(src, "w") as f:
        f.write('#include "route.h"\nusing namespace smk_route;\nextern "C" {\n' + declarations + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, src, "-o", lib], check=True)
    return ctypes.CDLL(lib)
