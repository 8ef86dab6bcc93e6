"""The device-memory pool and the pinned ring of the host-array calls
(csrc/host_mem.h), compiled for the CPU against a stand-in runtime whose
streams run as late as they may (tests/host_mem)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "host_mem")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_mem") / "host_mem_test")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", SRC,
                           "-I", os.path.join(ROOT, "imau-ice_amd", "csrc"),
                           os.path.join(SRC, "host_mem_test.cpp"), "-o", exe])
    return exe


@pytest.mark.parametrize("check", ["ring", "drop", "drop_of_another_thread", "threads", "reuse", "limit",
                                   "given_back", "out_of_memory", "closed", "pool_threads"])
def test_host_mem(program, check):
    r = subprocess.run([program, check], stdout=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
