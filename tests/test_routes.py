"""Host check (no GPU) of which kernel a call goes to, at sizes on both sides
of each line (tests/host/routes_check.cpp, linked with
voxtral.cpp_amd/csrc/vxfa_api.cpp)."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_calls_take_the_faster_kernel():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "routes_check")
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                            "-packed-fp32-ops", "-x", "hip", os.path.join(ROOT, "tests", "host", "routes_check.cpp"),
                            os.path.join(ROOT, "voxtral.cpp_amd", "csrc", "vxfa_api.cpp"), "-o", exe],
                           capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        env = {k: v for k, v in os.environ.items() if not k.startswith("VXFA_")}
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)
        assert r.returncode == 0 and r.stdout.startswith("ok"), (r.stdout + r.stderr)[-3000:]
