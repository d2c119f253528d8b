"""The FP32 prefilter drops no weighing sample of a splat near the spin axis, where an error of the pattern's phase moves
the sample further than the splat's centre. A host program built from the device headers
(tests/host/prefilter_axis_check.cpp) checks 200,000 samples around the cutoff."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_prefilter_keeps_weighing_samples_near_the_axis(tmp_path):
    exe = str(tmp_path / "prefilter_axis_check")
    src = os.path.join(HERE, "host", "prefilter_axis_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert "wrongly rejected 0" in out.stdout
