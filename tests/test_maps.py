"""The transfer's segment maps are bounded: a render groups its frames, a launch that cannot be split takes whole work
items. A host program built from the library's headers (tests/host/maps_check.cpp) checks the plans of launches from one
pixel to 4 million, in both precisions."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed to build the host check")
def test_maps_stay_within_their_limit(tmp_path):
    exe = str(tmp_path / "maps_check")
    src = os.path.join(HERE, "host", "maps_check.cpp")
    subprocess.run([HIPCC, "-O1", "--offload-arch=gfx950", "-x", "hip", "-w", "-o", exe, src], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
