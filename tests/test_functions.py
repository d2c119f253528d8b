"""The elementary functions of the transfer's coefficient fits: powers of one base from one logarithm, exp, log1p and
bounded sines are within 2 units of the last place of 64-bit-mantissa values and take the library's values at zero,
infinity and NaN. A host program built from the device headers (tests/host/fun_check.cpp) checks two million arguments."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_fit_functions_round_closely(tmp_path):
    exe = str(tmp_path / "fun_check")
    src = os.path.join(HERE, "host", "fun_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
