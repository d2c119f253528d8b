"""The transfer's FP32 prefilter is conservative: a sample at which a splat weighs above the cutoff is never dropped
before the pair queue, in either precision. A host program built from the device headers (tests/host/prefilter_check.cpp)
checks 200,000 samples around the cutoff of pattern and knot splats."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_prefilter_never_drops_a_weighing_splat(tmp_path):
    exe = str(tmp_path / "prefilter_check")
    src = os.path.join(HERE, "host", "prefilter_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert "wrongly rejected 0" in out.stdout
