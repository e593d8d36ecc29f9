"""CPU: the pool that keeps the eigensolve's device blocks between calls
(tests/workspace_check.cpp): bounded, one taker a block, given back when the
memory is short."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_block_pool(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "workspace_check")
    subprocess.check_call([gxx, "-O1", "-std=c++17", "-pthread", "-I",
                           os.path.join(ROOT, "nadvibs_amd", "csrc"),
                           os.path.join(ROOT, "tests", "workspace_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
