"""The FP64 PPM half-states on windows of special values (NaN, infinities, zeros, denormals, overflow),
compiled for the host from the device source, against the oracle's."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_ppm_half_states_of_special_values(tmp_path):
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    exe = tmp_path / "ppm_special_check"
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-x", "hip",
                    "-I" + os.path.join(ROOT, "chasqui_amd", "csrc"),
                    os.path.join(HERE, "native", "ppm_special_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "mismatches 0" in r.stdout, r.stdout + r.stderr
