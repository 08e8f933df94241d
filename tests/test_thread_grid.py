"""Launch grids of the tracer kernels with several threads per tracer, on the host:
from one tracer to the 2^31 - 1 an upload accepts, with 4 threads (samples, Heun, properties) and 9
(gradient rows scattered to upload order) each.  One axis of 2^24 blocks of 256 is
refused by the runtime, and 2^24 + 8 run as 8."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "dns_gkm_lpt_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not available")
def test_tracer_grids_stay_below_the_runtime_limit(tmp_path):
    exe = tmp_path / "thread_grid_check"
    subprocess.check_call([HIPCC, "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "host", "thread_grid_check.cpp"),
                           "-o", str(exe)], stdout=subprocess.DEVNULL)
    counts = [w * n for n in (1, 63, 64, 65, 10 ** 6, 2 ** 27 - 1, 2 ** 27, 2 ** 27 + 8, 2 ** 29 + 1, 2 ** 30, 2 ** 31 - 1)
              for w in (3, 4, 9)] + [2 ** 31, 2 ** 31 + 1]
    out = subprocess.run([str(exe)] + [str(n) for n in counts], capture_output=True, text=True, timeout=60)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
