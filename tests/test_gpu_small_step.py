"""The two-launch FP64 step of small grids (launch_small_step) against the three
sweeps and the CFL pass, which a context takes while its kernels are timed: same
expressions in the same order, so state and dt history are equal bit for bit.
Grids: the smallest, ones no tile divides, tile multiples, the largest."""
import numpy as np
import pytest

from cases import make_case
from dns_gkm_lpt_amd import _lib as gl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [16, 17, 31, 32, 63, 64, 96, 97])
def test_small_step_equals_sweeps(nc):
    W, P, _ = make_case(nc, seed=nc)
    out = []
    for timed in (False, True):
        with gl.Context(nc, P) as c:
            c.timing(timed)
            c.upload(W)
            dts = c.run(4, record_dt=True)
            c.step(float(dts[-1]))
            out.append((dts, c.cfl_dt(), c.download()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
    np.testing.assert_array_equal(out[0][2], out[1][2])


def test_dt_history_longer_than_the_device_keeps():
    """4096 dts are kept on the device between fetches."""
    W, P, _ = make_case(16)
    out = []
    for timed in (False, True):
        with gl.Context(16, P) as c:
            c.timing(timed)
            c.upload(W)
            out.append((c.run(4096, record_dt=True), c.run(4101, record_dt=True), c.run(1, record_dt=True), c.download()))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_small_step_reports_a_nonphysical_state():
    W, P, _ = make_case(32)
    W = W.copy()
    W[4][5, 6, 7] = -1.0
    with gl.Context(32, P) as c:
        c.upload(W)
        with pytest.raises(gl.GkmError) as e:
            c.run(2)
        assert e.value.code == 4


@pytest.mark.parametrize("compensate", [True, False])
@pytest.mark.parametrize("nc", [18, 20, 21, 32, 46, 100, 126, 128, 256])
def test_mixed_small_step_equals_sweeps(nc, compensate):
    """Mixed: first variants; state, carry and dt history bit for bit."""
    W, P, _ = make_case(nc, seed=nc)
    out = []
    for timed in (False, True):
        with gl.Context(nc, P, precision=gl.GKM_MIXED) as c:
            c.set_compensation(compensate)
            c.timing(timed)
            c.upload(W)
            dts = c.run(3, record_dt=True)
            c.step(float(dts[-1]))
            out.append((dts, c.cfl_dt(), c.download()) + ((c.download_carry(),) if compensate else ()))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nc", [112, 127, 160, 161])
def test_several_chunks_a_workgroup(nc):
    """Segments of more than one chunk, ragged and moved back into the grid."""
    test_small_step_equals_sweeps(nc)


@pytest.mark.parametrize("nc", [32, 50])
def test_mixed_context_with_other_tiles_keeps_its_sweeps(nc):
    W, P, _ = make_case(nc, seed=1)
    out = []
    for timed in (False, True):
        with gl.Context(nc, P, precision=gl.GKM_MIXED) as c:
            c.set_tiles((2, 1, 2))
            c.timing(timed)
            c.upload(W)
            c.run(3)
            out.append(c.download())
    np.testing.assert_array_equal(out[0], out[1])
