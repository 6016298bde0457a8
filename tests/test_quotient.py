"""Division by a number that the launch knows, on the host (no GPU): the library's own arithmetic (flash-dmattn_amd/csrc/fdma_params.h) is
compiled into tests/host/quotient_check.cpp with g++ and compared with the division of the language."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_quotients_are_exact_over_the_whole_range(tmp_path):
    exe = str(tmp_path / "quotient_check")
    cmd = ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I" + os.path.join(ROOT, "flash-dmattn_amd", "csrc"), os.path.join(ROOT, "tests", "host", "quotient_check.cpp"), "-o", exe]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().splitlines()[-1].startswith("OK"), run.stdout[-2000:]
