"""The host loops of the C ABI run every item once and pass an item's
exception on, with no, some or all of their threads started: a process at its
thread limit must not be aborted by a call that can do without them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ is not installed")
    exe = str(tmp_path_factory.mktemp("parallel") / "parallel_limits")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "grotor_amd", "csrc"),
                    os.path.join(ROOT, "tests", "parallel_limits.cpp"), "-o", exe, "-pthread", "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("threads", [0, 1, 3, 1000])
def test_loops_finish_with_any_number_of_threads(program, threads):
    r = subprocess.run([program, str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
