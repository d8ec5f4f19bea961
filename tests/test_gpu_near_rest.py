"""Flows near rest, where the HLLC flux's contact switch is a fraction on some
lanes of a wave and not on others, against the CPU oracle bit for bit."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd.ensemble import Ensemble
from pip_amd.solver import PIPSolver
from tests.util import interior

pytestmark = pytest.mark.gpu


def near_rest(flow, n, speed):
    """The flow's left state everywhere, with velocities of both fluids of
    either sign up to `speed` and zero in every third column."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    r = np.random.default_rng(n)
    out = []
    for u in (uh, um):
        u = u[:, :1, :1] + 0.0 * u
        m = u[0] * speed * r.standard_normal(u[1:4].shape)
        m[:, :, ::3] = 0.0
        rho = u[0]
        u[4] -= 0.5 * (u[1:4] ** 2).sum(0) / rho
        u[1:4] = m
        out.append(u)
    return cfg, out[0], out[1], ac


@pytest.mark.parametrize("speed", [1e-16, 1e-12, 3e-11])
@pytest.mark.parametrize("flow,n", [("orszag_tang", 40), ("kelvin_helmholtz", 40), ("orszag_tang", 300),
                                    ("brio_wu", 700)])
def test_runs_near_rest(flow, n, speed):
    cfg, uh, um, ac = near_rest(flow, n, speed)
    o = Oracle(cfg, uh, um, ac)
    o.run(nsteps=4)
    s = PIPSolver(cfg, uh, um, ac)
    s.advance(nsteps=4)
    for g, w in zip(s.state(), o.state()):
        assert np.array_equal(interior(g, cfg), interior(w, cfg))
    s.close()


@pytest.mark.parametrize("speed", [1e-13])
def test_sweep_near_rest(speed):
    """More 1-D tiles than CUs (264 of 255 cells)."""
    members = [near_rest("brio_wu", n, speed)[:3] for n in (30000, 300, 30000, 6600)]
    e = Ensemble(members, tend=1.0e30, max_steps=4, tile=256)
    e.set_mode("graph")
    e.run()
    for m, (cfg, uh, um) in enumerate(members):
        o = Oracle(cfg, uh, um, None)
        o.run(nsteps=4)
        for g, w in zip(e.state(m), o.state()):
            assert np.array_equal(interior(g, cfg), interior(w, cfg))
    e.close()
