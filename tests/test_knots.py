"""The knot interval of a trajectory splat: held at the first and last knot outside their times, finite where knot times
that ascend in FP64 coincide in FP32. A host program built from the device headers (tests/host/knot_check.cpp) checks it
against the sequential rule."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_knot_interval(tmp_path):
    exe = str(tmp_path / "knot_check")
    src = os.path.join(HERE, "host", "knot_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
