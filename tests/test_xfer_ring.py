"""The host side of field transfers (the pinned ring and its threads) on a
stand-in for the HIP runtime: every size and direction, from several threads,
from a thread whose current device is not the case's, beside other transfers
that stand still, and without pinned memory."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("xfer") / "xfer")
    stub = os.path.join(ROOT, "tests", "host_stub")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", stub, "-I", os.path.join(ROOT, "code_mge_amd", "csrc"),
                    "-o", exe, os.path.join(stub, "xfer_main.cpp")], check=True)
    return exe


@pytest.mark.parametrize("name", ["sizes", "threads", "device", "beside_one", "beside_five", "unpinned"])
def test_transfer(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
