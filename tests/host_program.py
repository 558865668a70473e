"""Builds the host programs of these tests against the library's internal header."""
import os
import subprocess

import gfirst_amd as ga

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "gfirst_amd")


def build(source, tmp_path):
    ga.lib()
    exe = str(tmp_path / os.path.splitext(source)[0])
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(LIB, "csrc"), "-I" + os.path.join(ROOT, "include"),
                    "-o", exe, os.path.join(HERE, source), "-L" + LIB, "-lgfirst",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + LIB], check=True)
    return exe
