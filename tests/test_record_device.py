"""An output thread's current GPU need not be the solver's: the record's
buffers are allocated and its kernel is launched on the solver's, and the
caller's current GPU is what it was."""
import os
import subprocess

import pytest

dyn = pytest.importorskip("dynfd3dcuda_amd")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "dynfd3dcuda_amd")


def test_record_on_the_solvers_gpu(tmp_path):
    dyn.load_library()
    exe = str(tmp_path / "record_device_tool")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"),
                           "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "record_device_tool.cpp"), "-o", exe,
                           "-rdynamic", "-L", PKG, "-lcgfdm", "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + PKG,
                           "-Wl,-rpath,/opt/rocm/lib", "-Wl,--allow-shlib-undefined"])
    assert subprocess.check_output([exe], text=True).split() == ["malloc", "1", "after", "0", "launch", "1", "after", "0"]
