"""Host check (no GPU) of the append launch's grid: voxtral.cpp_amd/csrc/
fa_kv_append.hip linked with a stand-in for the launch call
(tests/host/append_grid_check.cpp)."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_append_grid_covers_every_row_within_the_launch_limits():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "append_grid_check")
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                            "-packed-fp32-ops", "-x", "hip", os.path.join(ROOT, "tests", "host", "append_grid_check.cpp"),
                            os.path.join(ROOT, "voxtral.cpp_amd", "csrc", "fa_kv_append.hip"), "-o", exe],
                           capture_output=True, text=True, timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and r.stdout.startswith("ok"), (r.stdout + r.stderr)[-3000:]
