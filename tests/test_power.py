"""The power-law fits in FP32 stay finite where nu / nu_c passes FP32's range, and agree with FP64 where it does not. A host
program built from the device headers (tests/host/power_check.cpp) checks fields of 1e-24 to 1e21 G."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_power_law_fits_stay_finite(tmp_path):
    exe = str(tmp_path / "power_check")
    src = os.path.join(HERE, "host", "power_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
