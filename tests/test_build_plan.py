"""The plan of the builds by runs on the CPU (tests/plan/build_plan_check.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_accepted_sizes_have_room(tmp_path):
    exe = str(tmp_path / "build_plan_check")
    src = os.path.join(ROOT, "tests", "plan", "build_plan_check.cpp")
    cmd = [HIPCC, "--cuda-host-only", "-std=c++17", "-O1", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", src, "-o", exe]
    p = subprocess.run(cmd, capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "build plans ok" in r.stdout, r.stdout[-2000:]
