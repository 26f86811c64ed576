"""The engine's host side without a GPU: tests/cpp/engine_host_check.cpp brings a HIP runtime
of its own (device memory in host memory, launches only logged, allocations that fail on
demand), so that what the engine does when a call of the runtime fails is ordinary to check."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or no HIP headers")
    exe = str(tmp_path_factory.mktemp("engine") / "engine_host_check")
    lib = os.path.join(ROOT, "cellflow_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                    "-isystem", os.path.join(ROCM, "include"), "-I",
                    os.path.join(ROOT, "include"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "engine_host_check.cpp"),
                    "-L" + lib, "-lcellflow", "-Wl,-rpath," + lib], check=True)

    def run(case):
        out = subprocess.run([exe, case], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and f"{case} ok" in out.stdout, (out.returncode, out.stderr)

    return run


def test_failed_allocations_leave_the_sizes_true(check):
    check("grow_cells")


def test_state_changes_wait_for_their_kernels(check):
    check("changes_wait")


def test_copies_without_pinned_memory(check):
    check("pins_little")


def test_colours_after_a_failed_upload(check):
    check("colours")


def test_readback_with_another_device_current(check):
    check("other_device")


def test_long_rollout_needs_no_host_memory(check):
    check("long_rollout")
