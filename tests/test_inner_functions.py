"""The kernels' inner-loop functions and the split e-e-n polynomial, built for the
host against the emulation headers (tests/cpu_emu/inner_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_inner_functions_and_split_polynomial(tmp_path):
    exe = tmp_path / "inner_check"
    emu = os.path.join(HERE, "cpu_emu")
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", "-I" + os.path.join(emu, "include"), "-x", "c++",
                    os.path.join(emu, "inner_check.cpp"), "-x", "none", os.path.join(emu, "emu.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
