"""Host test of the layout of a Hamiltonian's coefficient block: the C++ test
program tests/c/test_coef_layout.cpp, linked against the library, with host
memory in the device's place."""
import os
import subprocess

import mcpi_amd
from mcpi_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_same_offsets_for_every_hamiltonian(tmp_path):
    lib = os.path.dirname(mcpi_amd.LIB_PATH)
    exe = str(tmp_path / "test_coef_layout")
    cmd = [build._hipcc(), *build.COMMON, "-I", os.path.join(ROOT, "mcpi_amd", "csrc"),
           os.path.join(ROOT, "tests", "c", "test_coef_layout.cpp"), "-L", lib,
           "-l:" + os.path.basename(mcpi_amd.LIB_PATH), "-Wl,-rpath," + lib, "-rdynamic", "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "all passed" in r.stdout
