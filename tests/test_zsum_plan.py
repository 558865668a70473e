"""The partials of the log-likelihood that a forward pass writes fit the buffer
made for them, whatever the geometry, the subset's length, the tile shape and the
chunks of the rotation; the kernel is one for all subsets of a subset count. On
the CPU: tests/zsum_plan_check.cpp asks the library's own launch plan."""
import os
import subprocess

import gfirst_amd as ga

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "gfirst_amd")


def build_host_program(source, exe):
    """Compiles a host program against the library's internal header."""
    ga.lib()
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(LIB, "csrc"), "-I" + os.path.join(ROOT, "include"),
                    "-o", exe, os.path.join(HERE, source), "-L" + LIB, "-lgfirst",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + LIB], check=True)
    return exe


def test_partials_fit_their_buffer(tmp_path):
    exe = build_host_program("zsum_plan_check.cpp", str(tmp_path / "zsum_plan_check"))
    out = subprocess.run([exe, "1000"], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    passes, narrow_short, cut, bad = map(int, out.stdout.split())
    # uneven subsets of narrow waves and cut chunks occur
    assert passes > 50_000 and narrow_short > 1000 and cut > 50 and bad == 0
