"""The ring of pinned buffers that large host copies go through (csrc/host_copy.hip),
on the host over a fake runtime (tests/host/fake_hip): bytes, a stream of another
device than the current one, failing copies, and no CPU time spent while the
stream's earlier work runs (0.5 s of it; the copy itself takes some 0.05 s of CPU,
eight threads spinning through it take 2 s or all the CPUs there are)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "dns_gkm_lpt_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_ring_over_a_fake_runtime(tmp_path):
    exe = tmp_path / "host_copy_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "host", "fake_hip"), "-I", CSRC,
                           "-x", "c++", os.path.join(CSRC, "host_copy.hip"), os.path.join(HERE, "host", "host_copy_check.cpp"),
                           "-o", str(exe), "-lpthread"])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
