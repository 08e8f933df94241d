"""The two-lane face flux (csrc/gkm_pair.hpp) and its two-lane reverse pass
(csrc/adj_pair.hpp) against the one-lane forms on the host, two threads standing
for the two lanes: 1500 seeded faces (air at 300 K, up to Mach 0.5, weak and
strong jumps).  Tolerances: 1e-12 of each flux component's largest magnitude and
1e-12 of the largest partial times its input, the bounds the one-lane forms are
held to against the oracle and against dual numbers (the two evaluate the same
terms in another order)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "dns_gkm_lpt_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not available")
def test_two_lane_forms_match_one_lane_forms(tmp_path):
    exe = tmp_path / "pair_check"
    subprocess.check_call([HIPCC, "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "host", "pair_check.cpp"),
                           "-o", str(exe), "-lpthread"], stdout=subprocess.DEVNULL)
    out = subprocess.run([str(exe), "1e-12", "1e-12"], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
