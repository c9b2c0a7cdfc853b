"""The cost model of the face march's segment (kernels.hpp march_seg), compiled for the host from the
device source, against the segments measured as good."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_march_segment_is_a_good_one(tmp_path):
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    exe = tmp_path / "march_seg_check"
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-x", "hip",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "chasqui_amd", "csrc"),
                    os.path.join(HERE, "native", "march_seg_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0 and "mismatches 0" in r.stdout, r.stdout + r.stderr
