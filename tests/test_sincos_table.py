"""The table variant of the k-space kernels' sin/cos, compiled for the host
from the kernels' header: within 1.3e-16 of long double (a table entry and the
last addition round by 2^-54 each at most, 1.11e-16, and the terms between them
are below 0.05 and round by a twentieth of that), and exactly periodic."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_sincos_table(tmp_path):
    exe = tmp_path / "sincos_table_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "rbmd_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "sincos_table_check.cpp"), "-o", str(exe)], check=True)
    e, differ = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert float(e) < 1.3e-16, e
    assert int(differ) == 0
