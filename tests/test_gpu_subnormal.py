"""Velocities and fields down among the subnormal numbers, as ahead of a front:
1-D runs and sweeps against the CPU oracle bit for bit, and 2-D runs the same
bits from every stage kernel.  (Below 2^-969 the kernels' quotients are not the
IEEE ones to the last bit, which 2-D runs at 1e-300 show against the oracle.)"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd.ensemble import Ensemble
from pip_amd.solver import PIPSolver
from tests.util import interior

pytestmark = pytest.mark.gpu


def faint(flow, n, size, fields):
    """A uniform state with momenta (and, with fields, B and psi instead of
    the flow's) of either sign about `size`, zero in every fifth column."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    r = np.random.default_rng(n)
    out = []
    for u in (uh, um):
        u = u[:, :1, :1] + 0.0 * u
        u[4] -= 0.5 * (u[1:4] ** 2).sum(0) / u[0]
        u[1:4] = size * r.standard_normal(u[1:4].shape)
        u[1:4, :, ::5] = 0.0
        out.append(u)
    if fields:
        um = out[1]
        um[4] -= 0.5 * (um[5:8] ** 2).sum(0)
        um[5:] = size * r.standard_normal(um[5:].shape)
        um[5:, :, ::5] = 0.0
    return cfg, out[0], out[1], ac


def oracle(cfg, uh, um, ac, steps):
    o = Oracle(cfg, uh, um, ac)
    o.run(nsteps=steps)
    return o.state()


def same(got, want, cfg):
    return all(np.array_equal(interior(g, cfg), interior(w, cfg)) for g, w in zip(got, want))


SIZES = [1e-322, 1e-316, 1e-308, 1e-306, 1e-300, 1e-290]


@pytest.mark.parametrize("fields", [False, True], ids=["velocities", "fields"])
@pytest.mark.parametrize("size", SIZES)
def test_1d_runs(size, fields):
    cfg, uh, um, ac = faint("brio_wu", 700, size, fields)
    s = PIPSolver(cfg, uh, um, ac)
    s.advance(nsteps=4)
    assert same(s.state(), oracle(cfg, uh, um, ac, 4), cfg)
    s.close()


# split tiles or, at 300^2, one-pass ones; other one-pass tiles; fluid by fluid
@pytest.mark.parametrize("fields", [False, True], ids=["velocities", "fields"])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("flow,n", [("orszag_tang", 40), ("orszag_tang", 300), ("kelvin_helmholtz", 40)])
def test_2d_kernels_agree(flow, n, size, fields):
    cfg, uh, um, ac = faint(flow, n, size, fields)
    ends = []
    for tile in ((16, 15, 1, 3), (16, 15, 1, 0), (16, 7, 1, 0), (32, 7, 0, 0)):
        s = PIPSolver(cfg, uh, um, ac, tile=tile)
        s.advance(nsteps=4)
        ends.append(s.state())
        s.close()
    for e in ends[1:]:
        assert same(e, ends[0], cfg)


@pytest.mark.parametrize("copies", [1, 100], ids=["few_tiles", "many_tiles"])
@pytest.mark.parametrize("size", [1e-322, 1e-316, 1e-308])
def test_sweeps(size, copies):
    cfg, uh, um, ac = faint("brio_wu", 700, size, False)
    e = Ensemble([(cfg, uh, um)] * copies, tend=1.0e30, max_steps=4, tile=256)
    e.set_mode("graph")
    e.run()
    assert same(e.state(copies - 1), oracle(cfg, uh, um, ac, 4), cfg)
    e.close()
