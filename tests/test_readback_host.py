"""The host logic of the threaded field copy (readback.hpp), compiled against a
double of the runtime's calls and run on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "channel_rl_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("readback") / "readback_check")
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "host"),
                    "-I", CSRC, os.path.join(HERE, "host", "readback_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["busy", "known", "memory"])
def test_readback(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
