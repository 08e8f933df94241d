"""The two-launch step of an ensemble against the three sweeps of each member
alone, which a context takes while its kernels are timed: same expressions in
the same order, so states are equal bit for bit.  Grids: the smallest, ragged
ones, tile multiples; a grid without the step (mixed: odd, or below its z tile)
sends the whole ensemble to the sweeps."""
import numpy as np
import pytest

from cases import make_case
from dns_gkm_lpt_amd import _lib as gl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,ncs", [
    (gl.GKM_FP64, (17, 48, 16, 33)),
    (gl.GKM_MIXED, (20, 64, 32, 50, 100)),
    (gl.GKM_MIXED, (32, 33)),
    (gl.GKM_MIXED, (32,)),
])
@pytest.mark.parametrize("graph", [False, True])
def test_ensemble_step_equals_members_sweeps(precision, ncs, graph):
    cs = [make_case(nc, seed=nc) for nc in ncs]
    alone = []
    for nc, (W, P, _) in zip(ncs, cs):
        with gl.Context(nc, P, precision=precision) as c:
            c.timing(True)
            c.upload(W)
            c.run(5)
            alone.append(c.download())
    with gl.Ensemble(list(ncs), [P for _, P, _ in cs], precision=precision) as e:
        for m, (W, _, _) in zip(e.members, cs):
            m.upload(W)
        e.run(2, graph=graph)
        e.run(3, graph=graph)
        for m, ref in zip(e.members, alone):
            np.testing.assert_array_equal(m.download(), ref)
