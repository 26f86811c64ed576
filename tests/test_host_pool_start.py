"""When the host threads of large loads and readbacks start and end
(tests/cpp/pool_start_check.cpp, CPU)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_threads_start_with_the_first_large_job(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = str(tmp_path / "pool_start_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "pool_start_check.cpp"),
                    os.path.join(ROOT, "cellflow_amd", "csrc", "cf_host.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "start ok" in out.stdout, (out.returncode, out.stderr)
