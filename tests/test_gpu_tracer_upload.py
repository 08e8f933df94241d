"""Tracers uploaded again: as many as before (the arrays stay), more, fewer, none.  A
context and an ensemble with captured graphs give what fresh ones give, bit for
bit."""
import numpy as np
import pytest

from cases import make_case
from dns_gkm_lpt_amd import _lib as gl
from dns_gkm_lpt_amd import ic as icm

pytestmark = pytest.mark.gpu


def outputs(c, dt):
    s = list(c.lpt_sample()) + [c.lpt_properties()]
    c.lpt_coupled_step(dt)
    return s + list(c.lpt_download())


def test_context_uploads_again():
    W, P, _ = make_case(32)
    sets = [icm.uniform_particles(n, seed=k) for k, n in enumerate((700, 700, 700, 65, 4000, 4000))]
    with gl.Context(32, P) as c:
        c.upload(W)
        dt = c.cfl_dt()
        for k, pos in enumerate(sets):
            c.upload(W)
            c.lpt_upload(pos)
            got = outputs(c, dt)
            with gl.Context(32, P) as f:
                f.upload(W)
                f.lpt_upload(pos)
                for a, b in zip(got, outputs(f, dt)):
                    np.testing.assert_array_equal(a, b)
            if k == 3:
                c.lpt_upload(np.zeros((0, 3)))
                with pytest.raises(gl.GkmError):  # no sample of the new tracers yet
                    c.lpt_upload(sets[0])
                    c.lpt_heun(dt)


def test_ensemble_uploads_again_between_graph_replays():
    cs = [make_case(nc, seed=nc) for nc in (32, 48)]
    a, b = icm.uniform_particles(500, seed=1), icm.uniform_particles(500, seed=2)

    def make():
        e = gl.Ensemble([32, 48], [P for _, P, _ in cs], precision=gl.GKM_MIXED)
        for m, (W, _, _) in zip(e.members, cs):
            m.upload(W)
        return e

    with make() as e:
        for m in e.members:
            m.lpt_upload(a)
        e.run(4, graph=True)
        for m, (W, _, _) in zip(e.members, cs):
            m.upload(W)
            m.lpt_upload(b)
        e.run(4, graph=True)
        got = [m.lpt_download() for m in e.members]
    with make() as e:
        for m in e.members:
            m.lpt_upload(b)
        e.run(4, graph=True)
        for m, (pos, vel) in zip(e.members, got):
            p, v = m.lpt_download()
            np.testing.assert_array_equal(pos, p)
            np.testing.assert_array_equal(vel, v)
