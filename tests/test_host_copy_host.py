"""csrc/host_copy.h without a GPU: compiled for the host over a stand-in for the HIP runtime (tests/host_copy), which runs the
copy kernels thread by thread and lets a test decide when, and which calls fail."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "bfuse-project_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_copy") / "test_host_copy")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wno-unused-function", "-pthread", "-I", os.path.join(HERE, "host_copy"), "-I", CSRC,
                    os.path.join(HERE, "host_copy", "test_host_copy.cc"), "-o", exe, "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("test", ["unaligned", "given_up", "arenas", "in_flight", "threads", "setup_fails"])
def test_host_copy(program, test):
    r = subprocess.run([program, test], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
