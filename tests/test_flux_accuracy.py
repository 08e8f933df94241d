"""Errors of the FP64 flux by two lanes per face (csrc/gkm_pair.hpp) and of its own
square root and exponential (csrc/gkm_math.hpp) against 80-bit values, on the host.

Bounds: a correctly rounded root is within half an ulp, 2^-53 = 1.1102e-16 of its
value: 1.12e-16.  The exponential: half an ulp of the sum for a result near
2^-1/2 (7.9e-17 of it), half an ulp of r <= ln 2 / 2 (2.8e-17) and three roundings
of terms of 0.06 (2.3e-17): 1.31e-16; the bound is the device exp's largest error,
1.35e-16.  The flux may be no further off than the one-lane form, component by
component, over 20000 seeded faces of uniform density and pressure and as many of a
developed flow."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "dns_gkm_lpt_amd", "csrc")
ORACLE = os.path.join(HERE, "..", "oracle")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not available")
def test_two_lane_flux_is_as_accurate_as_one_lane(tmp_path):
    exe = tmp_path / "accuracy_check"
    subprocess.check_call([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O2", "-mfma", "-fopenmp",
                           "-std=c++17", "-fpermissive", "-w", "-I", CSRC, "-I", ORACLE,
                           os.path.join(HERE, "host", "accuracy_check.cpp"), "-o", str(exe)])
    out = subprocess.run([str(exe), "1.12e-16", "1.35e-16"], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
