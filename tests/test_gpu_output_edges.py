"""Flow statistics and tracer properties at the edges of their kernels' parts:
grids whose columns fill no workgroup and whose lines are not multiples of the
16 cells a thread walks, tracer counts that leave a last wave with few quads.
Against the oracle, to the 1e-10 of test_gpu_lpt.py."""
import numpy as np
import pytest

import pyoracle as po
from cases import make_case
from dns_gkm_lpt_amd import _lib as gl
from dns_gkm_lpt_amd import ic as icm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,n", [(16, 1), (17, 63), (31, 65), (33, 257), (48, 1000)])
def test_statistics_and_properties(nc, n):
    W, P, gas = make_case(nc, seed=nc)
    pos = icm.uniform_particles(n, seed=nc)
    ref = po.field_stats(W, po.velocity_coefs(W), gas, P["p0"], P["Mt"], P["rho0"])
    rprops = po.particle_props(W, P["gam"], gas.dx, pos)
    with gl.Context(nc, P) as c:
        c.upload(W)
        s = c.stats()
        c.lpt_upload(pos)
        props = c.lpt_properties()
    pairs = [(s.tke, ref.tke), (s.diss, ref.diss), (s.sijsij, ref.sijsij), (s.enstrophy, ref.ens),
             (s.prms, ref.prms), (s.trms, ref.trms), (s.vrms, ref.vrms)]
    pairs += [(s.skew[a], ref.skew[a]) for a in range(3)] + [(s.kurt[a], ref.kurt[a]) for a in range(3)]
    for a, b in pairs:
        assert abs(a - b) <= 1e-10 * abs(b) + 1e-300, (a, b)
    # a column's scale: the flow's, where a single tracer's value may be near zero
    scale = np.maximum(np.max(np.abs(rprops), axis=0), 1e-300)
    many = np.max(np.abs(po.particle_props(W, P["gam"], gas.dx, icm.uniform_particles(500, seed=1))), axis=0)
    err = np.max(np.abs(props - rprops), axis=0) / np.maximum(scale, many)
    assert np.all(err < 1e-10), dict(zip(gl.PROP_NAMES, err))
