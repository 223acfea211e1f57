"""The staged state transfers (csrc/cs_transfer.h) on the host, over a fake of
the few runtime calls that they make (tests/fake_hip): what they do with
another device current, where staging fails, and for arrays and threads that
cannot be had."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not installed")
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-pthread", "-I", os.path.join(HERE, "fake_hip"), "-I",
                    os.path.join(ROOT, "cubesphere_amd", "csrc"), os.path.join(HERE, "transfer_check.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("what", ["first_small", "other_device", "fall_back", "pinned_arrays", "no_thread_memory"])
def test_transfer(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr[-300:])
