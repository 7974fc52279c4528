"""The prefix entries that the rect step kernel stages in LDS, with the code
that the kernel and the plan share, compiled for the CPU: never more than the
item's LDS holds, and all that its cells read."""

import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_staged_range_fits_its_lds(tmp_path):
    exe = str(tmp_path / "step_range_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror",
                    f"-I{REPO}/pyfstat_amd/csrc", f"-I{REPO}/include", "-o", exe,
                    os.path.join(REPO, "tests", "step_range_check.cpp")], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
