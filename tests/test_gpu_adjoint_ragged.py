"""The adjoint on grids whose 2 nc^3 lanes leave the flux adjoint's last workgroup
partly empty (csrc/adj_kernels.hip: lanes past the last face repeat it for the
exchange and store nothing): the dot-product identity <lam_N, dW_N> = <lam_0, dW_0>
with the tangent-linear run, which does not take that kernel, to test_gpu_adjoint.py's
1e-10; and lam_0 of a grid's cells translated periodically equals the translated
lam_0 to 1e-12 of its largest value per variable (the same terms summed in another
order of directions only at the wrap), so that the last faces carry what all do."""
import numpy as np
import pytest

from cases import make_case
from dns_gkm_lpt_amd import _lib as gl
from dns_gkm_lpt_amd import ic as icm

pytestmark = pytest.mark.gpu


def interior(a):
    nc = a.shape[-1] - 6
    return a[(slice(None),) + (slice(3, nc + 3),) * 3]


def padded(inner):
    nc = inner.shape[-1]
    v = np.zeros((5,) + (nc + 6,) * 3)
    v[(slice(None),) + (slice(3, nc + 3),) * 3] = inner
    return icm.fill_halo(v)


@pytest.mark.parametrize("nc", [16, 17, 20, 33])
def test_adjoint_with_a_ragged_last_workgroup(nc):
    W, P, _ = make_case(nc, seed=nc)
    scale = np.abs(interior(W)).max(axis=(1, 2, 3))[:, None, None, None]
    rng = np.random.default_rng(nc)
    dW0 = padded(1e-3 * scale * rng.standard_normal((5, nc, nc, nc)))
    lamN = padded(rng.standard_normal((5, nc, nc, nc)) / scale)
    move = (nc // 2, 3, nc - 5)
    roll = lambda a: padded(np.roll(interior(a), move, axis=(1, 2, 3)))
    with gl.Context(nc, P, precision=gl.GKM_FP64) as c:
        c.upload(W)
        dt = c.cfl_dt()
        dWN = c.tl_run(dt, 4, dW0)
        c.upload(W)
        lam0 = c.adjoint_run(dt, 4, 3, lamN)
        c.upload(roll(W))
        moved = c.adjoint_run(dt, 4, 3, roll(lamN))
    lhs = float(np.sum(interior(lamN) * interior(dWN)))
    rhs = float(np.sum(interior(lam0) * interior(dW0)))
    assert abs(lhs - rhs) <= 1e-10 * abs(lhs)
    ref = interior(roll(lam0))
    err = np.abs(interior(moved) - ref).max(axis=(1, 2, 3)) / np.abs(ref).max(axis=(1, 2, 3))
    print(nc, abs(lhs - rhs) / abs(lhs), err, flush=True)
    assert np.all(err <= 1e-12)
