"""No allocation that fails leaves a C entry as an exception (tests/host_entries.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc absent")
def test_no_exception_leaves_an_entry(tmp_path):
    exe = str(tmp_path / "host_entries")
    r = subprocess.run([HIPCC, "-std=c++17", "-O0", "-w", "--offload-arch=gfx950", "--offload-host-only",
                        "-Wl,--unresolved-symbols=ignore-all", "-x", "hip", "-I" + os.path.join(REPO, "include"),
                        "-I" + os.path.join(REPO, "porelb_amd", "csrc"), os.path.join(REPO, "tests", "host_entries.cpp"),
                        "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
