"""pip_time_steps runs and times the steps that pip_advance queues."""
import ctypes
import time

import numpy as np
import pytest

from pip_amd import problems
from pip_amd._lib import check, lib
from pip_amd.solver import PIPSolver

pytestmark = pytest.mark.gpu


def _run_ms(s, n):
    t = time.perf_counter()
    s.enqueue(n)
    s.sync()
    return (time.perf_counter() - t) * 1e3


def _total_ms(s, n):
    total = ctypes.c_double()
    check(lib().pip_time_steps(s.h, n, ctypes.byref(total), None, None))
    return total.value


@pytest.mark.parametrize("flow,n", [("brio_wu", 1024), ("orszag_tang", 64), ("orszag_tang", 300)])
def test_total_is_the_steps_own_time(flow, n):
    """Grids whose step ends run in the next step's first stage: a k_finalize
    of its own (4.5 us) or events between the launches (3.5 us each, three a
    step) would each be above 10 % of a step here."""
    s = PIPSolver(*getattr(problems, flow)(n))
    s.advance(nsteps=64)
    run = min(_run_ms(s, 128) for _ in range(5))
    total = min(_total_ms(s, 128) for _ in range(5))
    assert 0.5 * run < total < 1.1 * run, (total, run)
    s.close()


@pytest.mark.parametrize("stages", [True, False])
@pytest.mark.parametrize("flow,n", [("brio_wu", 200), ("orszag_tang", 40), ("orszag_tang", 500)])
@pytest.mark.parametrize("steps", [0, 1, 4, 7])
def test_steps_are_those_of_the_loop(steps, flow, n, stages):
    a = PIPSolver(*getattr(problems, flow)(n))
    b = PIPSolver(*getattr(problems, flow)(n))
    a.enqueue(steps)
    t = b.time_steps(steps, stages=stages)
    assert sorted(t) == (["stage1_ms", "stage2_ms", "total_ms"] if stages else ["total_ms"])
    if stages and steps:
        assert 0.0 < t["stage1_ms"] and 0.0 < t["stage2_ms"] and t["stage1_ms"] + t["stage2_ms"] < t["total_ms"]
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)
    assert a.scalars() == b.scalars()
    for s in (a, b):
        s.close()
