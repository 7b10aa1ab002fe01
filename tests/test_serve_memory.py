"""The RSQF serving loop's memory on a model of the device (no GPU;
tests/plan/serve_check.cpp): gather buffers, workers kept between runs, the
budget."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    exe = str(tmp_path_factory.mktemp("serve") / "serve_check")
    src = os.path.join(ROOT, "tests", "plan", "serve_check.cpp")
    cmd = [HIPCC, "--cuda-host-only", "-std=c++17", "-O1", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", src, "-o", exe, "-lpthread",
           "-Wl,--unresolved-symbols=ignore-all"]  # (the device code that the launch stubs name)
    p = subprocess.run(cmd, capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-3000:]
    return exe


@pytest.mark.parametrize("scenario", ["exact", "refused", "idle"])
def test_serving_memory(check, scenario):
    r = subprocess.run([check, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and scenario + " ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
