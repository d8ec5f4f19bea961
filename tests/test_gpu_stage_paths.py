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
