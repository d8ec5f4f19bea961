"""Runs that stop inside a chunk of queued steps: what the chunk's other steps
cost, and that they leave the state, the scalars and a recorded history alone."""
import ctypes
import time

import numpy as np
import pytest
import torch

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd._lib import check, lib
from pip_amd.solver import PIPSolver
from tests.util import interior

pytestmark = pytest.mark.gpu


def _us_per_step(s, n, tend=1.0e300):
    best = 1.0e30
    for _ in range(3):
        t = time.perf_counter()
        s.enqueue(n, tend)
        s.sync()
        best = min(best, (time.perf_counter() - t) / n)
    return best * 1e6


@pytest.mark.parametrize("flow,n", [("orszag_tang", 1024), ("kelvin_helmholtz", 1500)])
def test_steps_of_a_stopped_run_are_cheap(flow, n):
    """A stopped run's steps are three launches that look at a flag (2 to 8 us
    each with their workgroups' starts), where a running step of these sizes
    takes 250 us and more: under a tenth of it, and over it if they read the
    state (a third to a fifth of a step's bytes)."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    s = PIPSolver(cfg, uh, um, ac)
    s.advance(nsteps=4)
    running = _us_per_step(s, 16)
    s.advance(tend=s.scalars()["time"] + 0.5 * s.scalars()["dt"])
    s.enqueue(1, s.scalars()["time"])  # the loop's top finds the end reached
    nt = s.scalars()["nt"]
    stopped = _us_per_step(s, 64)
    assert s.scalars()["nt"] == nt
    assert stopped < 0.1 * running, (stopped, running)
    s.close()


# step ends folded into split tiles, into one-pass tiles (361 of 16x15), not
# folded; the fluid-by-fluid kernel; 1-D
PATHS = [("orszag_tang", 40, (16, 7, 1, 0)), ("kelvin_helmholtz", 300, (16, 15, 1, 0)),
         ("orszag_tang", 420, (16, 15, 1, 0)), ("orszag_tang", 40, (16, 15, 1, 3)), ("brio_wu", 300, None)]


@pytest.mark.parametrize("flow,n,tile", PATHS)
def test_stop_inside_a_chunk(flow, n, tile):
    """An end time in a chunk's third step, and on again."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    o = Oracle(cfg, uh, um, ac)
    s = PIPSolver(cfg, uh, um, ac, tile=tile)
    tend = 2.5 * s.scalars()["dt"]
    o.run(tend=tend)
    s.advance(tend=tend)
    assert (s.scalars()["nt"], s.scalars()["time"]) == (o.scalars()["nt"], o.scalars()["time"])
    o.run(nsteps=2)
    s.advance(nsteps=2)
    for g, w in zip(s.state(), o.state()):
        assert np.array_equal(interior(g, cfg), interior(w, cfg))
    so, sg = o.scalars(), s.scalars()
    assert (sg["dt"], sg["time"], sg["nt"]) == (so["dt"], so["time"], so["nt"])
    s.close()


@pytest.mark.parametrize("flow,n,tile", PATHS)
def test_recorded_history_past_a_stop(flow, n, tile):
    """A recorded run stops on a NaN after its first step: the history's other
    steps hold dt = 0 and the last GLM speed, whatever the chunk's length."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    um[6, um.shape[1] // 2, um.shape[2] // 2] = np.nan
    for steps in (1, 2, 5, 6):
        s = PIPSolver(cfg, uh, um, ac, tile=tile)
        hist = torch.full((2 * steps,), -1.0, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        check(lib().pip_record_steps(s.h, steps, ctypes.c_void_p(hist.data_ptr())))
        s.sync()
        h = hist.cpu().numpy().reshape(steps, 2)
        assert s.scalars()["nt"] == 1 and s.status() == 2
        assert h[0, 0] > 0.0 and not h[1:, 0].any() and (h[:, 1] == h[0, 1]).all()
        s.close()
