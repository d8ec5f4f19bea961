"""The paths the stage kernels and the step loop choose by size and state,
against the CPU oracle bit for bit, at the sizes where the choice changes."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd.solver import PIPSolver
from tests.util import interior

pytestmark = pytest.mark.gpu


def same_as_oracle(cfg, uh, um, ac, nsteps, tile=None):
    o = Oracle(cfg, uh, um, ac)
    o.run(nsteps=nsteps)
    s = PIPSolver(cfg, uh, um, ac, tile=tile)
    s.advance(nsteps=nsteps)
    oh, om = o.state()
    gh, gm = s.state()
    assert np.array_equal(interior(gm, cfg), interior(om, cfg))
    assert np.array_equal(interior(gh, cfg), interior(oh, cfg))
    so, sg = o.scalars(), s.scalars()
    assert (sg["dt"], sg["time"], sg["nt"]) == (so["dt"], so["time"], so["nt"])
    s.close()


@pytest.mark.parametrize("flow", ["orszag_tang", "kelvin_helmholtz"])
@pytest.mark.parametrize("n", [120, 121, 500])
def test_reduction_slot_sets(flow, n):
    """dt from 1, 2 and 16 sets of reduction slots (64, 72 and 1088 tiles)."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    same_as_oracle(cfg, uh, um, ac, nsteps=3)


@pytest.mark.parametrize("power", [98, 104])
@pytest.mark.parametrize("flow,n", [("orszag_tang", 47), ("kelvin_helmholtz", 33)])
def test_states_beyond_the_bounded_range(flow, n, power):
    """Densities and pressures at and above 2^100, where the stage takes the
    general fluxes (the same flow in other units of mass: B scales by the
    root, so power is even; flag_IR 0, as the rates are not scale-free)."""
    cfg, uh, um, _ = getattr(problems, flow)(n)
    um[:5] *= 2.0 ** power
    uh *= 2.0 ** power
    um[5:8] *= 2.0 ** (power // 2)
    same_as_oracle(cfg.replace(flag_ir=0, col=cfg.col * 2.0 ** -power), uh, um, None, nsteps=20)
