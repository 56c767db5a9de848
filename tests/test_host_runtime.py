"""The runtime's host side (fivonagi_amd/csrc/fv_runtime.cpp) on a stand-in for
the HIP runtime: what it launches, copies and waits for (tests/host)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "fivonagi_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = tmp_path_factory.mktemp("host") / "runtime_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "host"),
                    "-o", str(exe), os.path.join(HERE, "host", "runtime_check.cpp"),
                    os.path.join(CSRC, "fv_runtime.cpp"), os.path.join(CSRC, "fv_tables.cpp")],
                   check=True)
    return str(exe)


@pytest.mark.parametrize("name", [
    "collect_without_ring", "download_error", "download_device",
    "enqueue_under_capture", "autotune", "no_pinned_memory",
])
def test_runtime(check, name):
    r = subprocess.run([check, name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
