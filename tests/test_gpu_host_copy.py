"""Copies of whole arrays through the pinned ring (csrc/host_copy.hip): sizes
below and just above the 32 MB at which it starts, tails that fill no slice, several
segments, several contexts at once.  Bytes have to arrive as they are."""
import ctypes
import threading

import numpy as np
import pytest

from cases import make_case
from dns_gkm_lpt_amd import _lib as gl
from dns_gkm_lpt_amd import ic as icm

pytestmark = pytest.mark.gpu
PAR = dict(gam=1.4, mu0=1e-3, p0=86100.0)


def random_state(nc, seed):
    return icm.fill_halo(np.random.default_rng(seed).standard_normal((5, nc + 6, nc + 6, nc + 6)))


@pytest.mark.parametrize("nc", [87, 89, 101, 160])  # 32.2 MB (plain), 34.3, 49, 183 MB
def test_state_round_trip(nc):
    W = random_state(nc, nc)
    with gl.Context(nc, PAR) as c:
        for k in range(2):  # the second pass reuses the ring
            c.upload(W + k)
            np.testing.assert_array_equal(c.download(), W + k)


def test_contexts_in_threads():
    states = [random_state(96, s) for s in range(3)]
    got = [None] * 3

    def work(m):
        with gl.Context(96, PAR) as c:
            for _ in range(3):
                c.upload(states[m])
                got[m] = c.download()

    threads = [threading.Thread(target=work, args=(m,)) for m in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m in range(3):
        np.testing.assert_array_equal(got[m], states[m])


def test_tracer_arrays_in_parts():
    """np x 9 gradients split into the three arrays (33.6 MB, three segments), and
    np x 41 properties (153 MB), against each other: the same splines evaluated
    by two kernels, equal to 1e-12 of the largest gradient (about 100 roundings of
    64-term sums)."""
    n = 466_667
    W, P, _ = make_case(32)
    pos = icm.uniform_particles(n, 3)
    with gl.Context(32, P) as c:
        c.upload(W)
        c.lpt_upload(pos)
        U, gU, gV, gW = c.lpt_sample()
        props = c.lpt_properties()
    for a, b in ((U, props[:, 1:4]), (gU, props[:, 8:11]), (gV, props[:, 11:14]), (gW, props[:, 14:17])):
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))


@pytest.mark.parametrize("nc", [64, 101])
def test_pinned_memory_goes_straight(nc):
    """Memory the runtime knows takes the plain copy on both sides of the 32 MB."""
    W = random_state(nc, nc)
    with gl.Context(nc, PAR) as c:
        hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime the library loaded
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(W.nbytes), 0) == 0
        pinned = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), W.shape)
        pinned[:] = W
        c.upload(pinned)
        np.testing.assert_array_equal(c.download(), W)
        assert hip.hipHostFree(p) == 0
