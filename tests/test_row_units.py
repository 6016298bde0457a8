"""Which block of query rows a workgroup of the forward and of dQ has, on the host (no GPU): the library's own mapping
(flash-dmattn_amd/csrc/fdma_params.h) is compiled into tests/host/row_units_check.cpp with g++ and swept over batches of one length and
ragged ones."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_block_has_one_workgroup_and_launches_are_not_mostly_empty(tmp_path):
    exe = str(tmp_path / "row_units_check")
    cmd = ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I" + os.path.join(ROOT, "flash-dmattn_amd", "csrc"), os.path.join(ROOT, "tests", "host", "row_units_check.cpp"), "-o", exe]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().splitlines()[-1].startswith("OK"), run.stdout[-2000:]
