"""A context and an ensemble where the two-launch step's memory is not to be had:
they are made without it, as they were before there was one, and step by the sweeps
to the same bits.  hipMalloc is stood in for by one that fails for what does not fit
a budget, in a process of its own; what the library asks for is measured first."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

INTERPOSER = r"""
#include <dlfcn.h>
#include <cstddef>
#include <map>
static std::map<void*, size_t> held;
static size_t budget = ~(size_t)0, used = 0, peak = 0;
template <typename F> static F real(const char* n)
{
    static void* hip = dlopen("libamdhip64.so", RTLD_NOW | RTLD_NOLOAD);
    static void* any = hip ? hip : dlopen(HIP_LIBRARY, RTLD_NOW);
    return (F)dlsym(any, n);
}
extern "C" void set_budget(size_t b) { budget = b; peak = used; }
extern "C" size_t peak_use() { return peak; }
extern "C" int hipMalloc(void** p, size_t n)
{
    if (used + n > budget) return 2;  // hipErrorOutOfMemory
    static auto f = real<int (*)(void**, size_t)>("hipMalloc");
    const int rc = f(p, n);
    if (rc == 0) held[*p] = n, used += n, peak = used > peak ? used : peak;
    return rc;
}
extern "C" int hipFree(void* p)
{
    auto it = held.find(p);
    if (it != held.end()) used -= it->second, held.erase(it);
    static auto f = real<int (*)(void*)>("hipFree");
    return f(p);
}
"""

CHILD = r"""
import ctypes, sys
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/../oracle", sys.argv[2] + "/.."]
import numpy as np
lib = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib.peak_use.restype = ctypes.c_size_t
lib.set_budget.argtypes = [ctypes.c_size_t]
from cases import make_case
from dns_gkm_lpt_amd import _lib as gl

W, P, _ = make_case(48)

def context(prec):
    with gl.Context(48, P, precision=prec) as c:
        c.upload(W)
        c.run(3)
        return c.download()

def ensemble(prec):
    with gl.Ensemble([48] * 3, [P] * 3, precision=prec) as e:
        for m in e.members:
            m.upload(W)
        e.run(3)
        return np.stack([m.download() for m in e.members])

extra = (15 - 5) * 48 ** 3 * 8 - 5 * 54 ** 3 * 8  # the face fluxes past dW and the staging area
assert extra > 0
for prec in (gl.GKM_FP64, gl.GKM_MIXED):
    for make, members in ((context, 1), (ensemble, 3)):
        lib.set_budget(2 ** 40)
        ref = make(prec)
        full = lib.peak_use()
        for short in (1, members * extra - 4096 * members):
            lib.set_budget(full - short)
            np.testing.assert_array_equal(make(prec), ref)
            print("ok", prec, members, full, short, flush=True)
        lib.set_budget(full - members * extra - (1 << 20))
        try:
            make(prec)
        except gl.GkmError as err:
            assert err.code == 3, err.code
        else:
            raise AssertionError("a budget below the old need was enough")
print("all right")
"""


def test_two_launch_memory_is_optional(tmp_path):
    from dns_gkm_lpt_amd import _lib
    ldd = subprocess.run(["ldd", _lib.LIB_PATH], capture_output=True, text=True).stdout
    hip = next(line.split("=>")[1].split()[0] for line in ldd.splitlines() if "libamdhip64" in line and "=>" in line)
    src, so, child = tmp_path / "budget.cpp", tmp_path / "budget.so", tmp_path / "child.py"
    src.write_text(INTERPOSER)
    child.write_text(CHILD)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-DHIP_LIBRARY=\"%s\"" % hip, str(src), "-o",
                           str(so), "-ldl"])
    out = subprocess.run([sys.executable, str(child), str(so), HERE], capture_output=True, text=True, timeout=100)
    print(out.stdout, out.stderr[-2000:])
    assert out.returncode == 0 and out.stdout.strip().endswith("all right")
