"""The start of 2-D ensembles of very uneven sizes."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd.ensemble import Ensemble
from tests.util import interior

pytestmark = pytest.mark.gpu


def _members(n_small, n_large, large):
    return [problems.orszag_tang(4)[:3]] * n_small + [problems.orszag_tang(large)[:3]] * n_large


def test_many_small_members_and_a_large_one():
    """5000 members of 4 x 4 cells leave 16 workgroups a member, which go over
    the large one's 92,416 cells 23 times."""
    e = Ensemble(_members(5000, 1, 300), tend=1.0e30, max_steps=3)
    e.set_mode("graph")
    e.run()
    for m in (0, 2500, 5000):
        cfg, uh, um = _members(1, 1, 300)[m == 5000]
        o = Oracle(cfg, uh, um, None)
        o.run(nsteps=3)
        for g, w in zip(e.state(m), o.state()):
            assert np.array_equal(interior(g, cfg), interior(w, cfg))
        assert e.result(m)["time"] == o.scalars()["time"]
    e.close()


def test_start_costs_what_the_members_need():
    """Runs that end where they start: the start of both kinds together takes less than
    twice that of each alone (with a workgroup per 256 cells of the largest for
    every member, 41 million, several times as long)."""
    ms = []
    for n_small, n_large in ((5000, 0), (0, 1), (5000, 1)):
        e = Ensemble(_members(n_small, n_large, 1024), tend=0.0, max_steps=1)
        e.set_mode("graph")
        e.run()
        t = []
        for _ in range(4):
            e.reset()
            t.append(e.run())
        ms.append(min(t))
        e.close()
    assert ms[2] < 2.0 * (ms[0] + ms[1]), ms
