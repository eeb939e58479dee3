"""Workgroups per compute unit limited through LDS (voreen_amd/csrc/residency.h,
batched launches' `resident`): exactly the asked number fits for every static
LDS size, checked on the host by tests/native/residency_check.cpp, compiled
from the header that the launches include.  CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_exactly_the_asked_number_fits(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "residency_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "voreen_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "residency_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
