"""Host code of the transfers and of the kept device blocks, on a HIP runtime
made of malloc (tests/host_memory.cpp), under the address sanitizer."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

INCLUDE = "/opt/rocm/include"


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(INCLUDE, "hip")):
        pytest.skip("g++ or the HIP headers absent")
    out = str(tmp_path_factory.mktemp("host") / "host_memory")
    csrc, tests = os.path.join(REPO, "porelb_amd", "csrc"), os.path.join(REPO, "tests")
    sources = [os.path.join(tests, "host_memory.cpp"), os.path.join(csrc, "plb_mem.hip"), os.path.join(csrc, "plb_xfer.hip")]
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined", "-w",
                        "-D__HIP_PLATFORM_AMD__", "-include", os.path.join(tests, "host_hip.hpp"), "-I" + INCLUDE,
                        "-I" + os.path.join(REPO, "include"), "-I" + csrc, "-x", "c++", *sources, "-o", out],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("check", ["device", "at_exit", "release", "room"])
def test_host_memory(exe, check):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "ERROR" not in r.stderr and "runtime error" not in r.stderr, r.stderr
