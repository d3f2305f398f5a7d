"""The rules that give an on-chip plan its shape and its kernel agree, for every
block size and LDS size (host code only, tests/host_onchip.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc absent")
def test_plan_and_kernel_agree(tmp_path):
    exe = str(tmp_path / "host_onchip")
    r = subprocess.run([HIPCC, "-std=c++17", "-O0", "-w", "--offload-arch=gfx950", "--offload-host-only", "-Wl,--unresolved-symbols=ignore-all", "-x", "hip",
                        "-I" + os.path.join(REPO, "include"), "-I" + os.path.join(REPO, "porelb_amd", "csrc"),
                        os.path.join(REPO, "tests", "host_onchip.cpp"), "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
