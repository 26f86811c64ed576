"""The host threads of large loads and readbacks: when they start and end
(tests/cpp/pool_start_check.cpp), and both of the pool's programs under the thread, address and
undefined-behaviour sanitizers (CPU)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "cellflow_amd", "csrc", "cf_host.cpp")


def compile_run(exe, sources, flags):
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", *flags, "-o", exe, *sources],
                   check=True, stderr=subprocess.DEVNULL)
    # the sanitizers' runtimes need not come first among preloaded libraries
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    return subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)


@pytest.mark.parametrize("sanitizer", ["", "thread", "address,undefined"])
@pytest.mark.parametrize("program", ["pool_start_check", "pool_check"])
def test_threads(tmp_path, program, sanitizer):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    flags = ["-fsanitize=" + sanitizer] if sanitizer else []
    if sanitizer:  # the sanitizer has to work at all on this machine
        empty = tmp_path / "empty.cpp"
        empty.write_text("int main() { return 0; }\n")
        try:
            if compile_run(str(tmp_path / "empty"), [str(empty)], flags).returncode != 0:
                pytest.skip(f"-fsanitize={sanitizer} does not run here")
        except subprocess.CalledProcessError:
            pytest.skip(f"no -fsanitize={sanitizer}")
    out = compile_run(str(tmp_path / program),
                      [os.path.join(ROOT, "tests", "cpp", program + ".cpp"), HOST], flags)
    said = {"pool_start_check": "start ok", "pool_check": "pool ok"}[program]
    assert out.returncode == 0 and said in out.stdout and "Sanitizer" not in out.stderr, \
        (out.returncode, out.stderr[-3000:])
