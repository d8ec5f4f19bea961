"""The paths the stage kernels and the step loop choose by size and state,
against the CPU oracle bit for bit, at the sizes where the choice changes."""
import ctypes

import numpy as np
import pytest
import torch

from oracle.oracle import Oracle
from pip_amd import problems
from pip_amd._lib import check, lib
from pip_amd.adjoint import TwoFluidRun
from pip_amd.config import PIPConfig
from pip_amd.ensemble import Ensemble
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


def cut(flow, nx, ny, **kw):
    """An nx x ny corner of a flow's square grid, same cell size."""
    n = max(nx, ny)
    cfg, uh, um, _ = getattr(problems, flow)(n)
    kw.update(nx=nx, ny=ny, xmax=cfg.xmin + nx * cfg.dx, ymax=cfg.ymin + ny * cfg.dy)
    sl = (slice(None), slice(0, ny + 4), slice(0, nx + 4))
    return cfg.replace(**kw), uh[sl].copy(), um[sl].copy(), None


# default tiles: 16x7 split while they number at most 256, then 16x15 split
# while those do, then 16x15 one-pass
SIZES = [(4, 4), (16, 7), (17, 8), (33, 20), (256, 112), (257, 112), (256, 240), (257, 240)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("flow,kw", [
    ("orszag_tang", {}),
    ("kelvin_helmholtz", {}),
    ("orszag_tang", dict(t_order=3, flag_bnd=(10, 10, 2, 10))),
    ("orszag_tang", dict(flag_col=5, col=5.0, flag_pip_imp=1)),
    ("kelvin_helmholtz", dict(flag_col=4, col=5.0, flag_pip_imp=1)),
    ("kelvin_helmholtz", dict(flag_divb=0, flag_ir_type=1)),
], ids=["plain", "ir", "rk3_outflow", "col_imp", "ir_col_imp", "no_psi"])
def test_split_tiles(nx, ny, flow, kw):
    """Each path the stage takes by grid size, at the sizes where it changes
    and at partial tiles, with every option its cell phase splits over."""
    cfg, uh, um, ac = cut(flow, nx, ny, **kw)
    if kw.get("flag_divb") == 0:
        um = um[:8].copy()
    same_as_oracle(cfg, uh, um, ac, nsteps=3 if nx * ny > 20000 else 8)


@pytest.mark.parametrize("nx", [4, 127, 128, 1000, 127 * 256, 127 * 256 + 1])
@pytest.mark.parametrize("kw", [{}, dict(flag_ir=3), dict(flag_col=2, col=5.0, flag_pip_imp=1, t_order=3)],
                         ids=["plain", "ir", "col_imp_rk3"])
def test_split_tiles_1d(nx, kw):
    cfg, uh, um, ac = problems.brio_wu(nx)
    same_as_oracle(cfg.replace(**kw), uh, um, ac, nsteps=8)


@pytest.mark.parametrize("n", [20, 200])
@pytest.mark.parametrize("tile", [(16, 7), (16, 15)])
def test_split_tiles_in_the_adjoints_runs(n, tile):
    """Recorded and replayed steps (16x7 and 16x15 split, one-pass beyond)
    end where the plain run does, saved inputs and primitives included."""
    cfg, uh, um, ac = problems.alfven_damping(n)
    u0 = torch.from_numpy(np.concatenate([um, uh])).cuda()
    act = torch.from_numpy(ac).cuda()
    ends = []
    for t, keep in ((tile + (1, 0), 2), ((32, 7, 1, 0), 0)):
        r = TwoFluidRun(cfg, nsteps=6, ckpt_every=2, tile=t, replay_tile=t, keep_segments=keep)
        a, b = u0.clone().requires_grad_(), act.clone().requires_grad_()
        out = r.run(a, b)
        g = torch.autograd.grad((out[:, 2:-2, 2:-2] ** 2).sum(), (a, b))
        ends.append((out.detach(), *g, r.replay(u0, act)))
        r.close()
    for x, y in zip(*ends):
        assert torch.equal(x, y)


@pytest.mark.parametrize("flow,n", [("brio_wu", 300), ("orszag_tang", 24), ("kelvin_helmholtz", 20)])
def test_folded_step_ends(flow, n):
    """On split grids a step's end runs in the next step's first stage: chunks
    of odd and even lengths, a run that stops on its end time inside a chunk
    and goes on, and the procedures in between, against the oracle."""
    cfg, uh, um, ac = getattr(problems, flow)(n)
    o = Oracle(cfg, uh, um, ac)
    s = PIPSolver(cfg, uh, um, ac)
    for steps in (1, 2, 3, 64, 65, 128):
        o.run(nsteps=steps)
        assert s.advance(nsteps=steps)[0] == steps
        assert (s.scalars()["dt"], s.scalars()["time"]) == (o.scalars()["dt"], o.scalars()["time"])
    tend = o.scalars()["time"] + 20.5 * o.scalars()["dt"]
    o.run(tend=tend)
    s.advance(tend=tend)
    assert s.scalars()["nt"] == o.scalars()["nt"]
    o.run(nsteps=5)
    s.advance(nsteps=5)
    oh, om = o.state()
    gh, gm = s.state()
    assert np.array_equal(interior(gm, cfg), interior(om, cfg)) and np.array_equal(interior(gh, cfg), interior(oh, cfg))
    assert (s.scalars()["dt"], s.scalars()["time"]) == (o.scalars()["dt"], o.scalars()["time"])
    # a NaN stops the run at its step's end and is still flagged after it
    um[6, um.shape[1] // 2, um.shape[2] // 2] = np.nan
    b = PIPSolver(cfg, uh, um, ac)
    assert b.advance(nsteps=70)[0] == 1 and b.status() == 2
    for x in (s, b):
        x.close()


@pytest.mark.parametrize("n", [33, 300])
def test_ionisation_rates_that_underflow(n):
    """Plasma from its own temperature down to where the ionisation rate passes
    1e-250 (a = 13.6 eV / T near 570) and then zero (near 740)."""
    cfg, uh, um, ac = problems.kelvin_helmholtz(n)
    rest = 0.5 * (um[1:4] ** 2).sum(0) / um[0] + 0.5 * (um[5:8] ** 2).sum(0)
    colder = np.geomspace(1.0, 1.0 / 40.0, um.shape[2])
    um[4] = (um[4] - rest) * colder + rest
    same_as_oracle(cfg, uh, um, ac, nsteps=3)


@pytest.mark.parametrize("nx,ny", [(4, 4), (8, 8), (9, 17), (65, 48), (128, 128), (129, 128), (40, 523)])
@pytest.mark.parametrize("bnd", [(1, 1, 1, 1), (2, 2, 3, 2)], ids=["periodic", "mirror"])
def test_adjoint_gathers(nx, ny, bnd):
    """One adjoint step on 8 x 8 gather tiles (up to 256 of them) and on
    16 x 13 ones against the host build of the work items, at the bar of
    test_adjoint_step_equals_host_work_items."""
    from tests.test_adjoint_cpu import L as host, _smooth_state
    cfg = PIPConfig(ndim=2, nx=nx, ny=ny, xmin=0.0, xmax=1.0, ymin=0.0, ymax=ny / nx, flag_divb=1, ac_field=True,
                    flag_bnd=bnd, col=30.0)
    o = Oracle(cfg, *_smooth_state(cfg, 5), prologue=False)
    o.pipbnd()
    uh, um = o.state()
    ac = _smooth_state(cfg, 5)[2]
    dt = 0.05 * min(cfg.dx, cfg.dy)
    cmax = cfg.safety * min(cfg.dx, cfg.dy) / dt
    o.set_scalars(dt, cmax)
    U1 = np.ascontiguousarray(o.run_solver_stage1())
    U = np.ascontiguousarray(np.concatenate([um, uh]))
    W = np.random.default_rng(17).normal(size=U.shape)
    lam_h, lam_ac_h = W.copy(), np.zeros((cfg.jx, cfg.ix))
    P, I = ctypes.POINTER(ctypes.c_double), ctypes.c_int
    host.hc_adj_step.argtypes = [I, I, P, ctypes.POINTER(I), P, P, P, P, P]
    prm = np.array([cfg.gm, cfg.ro_lim, cfg.pr_lim, cfg.dx, cfg.dy, cfg.col, cfg.safety, cfg.db_clean, dt, cmax])
    host.hc_adj_step(cfg.ix, cfg.jx, prm.ctypes.data_as(P), (I * 4)(*bnd),
                     *(x.ctypes.data_as(P) for x in (U, U1, np.ascontiguousarray(ac), lam_h, lam_ac_h)))
    s = PIPSolver(cfg, uh, um, ac, prologue=False)
    Ud, U1d, lam = (torch.tensor(x, device="cuda:0") for x in (U, U1, W))
    dtc = torch.tensor([dt, cmax], dtype=torch.float64, device="cuda:0")
    lam_ac = torch.zeros((cfg.jx, cfg.ix), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    check(lib().pip_adj_seed(s.h, lam.data_ptr()))
    check(lib().pip_adj_step(s.h, Ud.data_ptr(), U1d.data_ptr(), None, None, dtc.data_ptr(), lam.data_ptr(),
                             lam_ac.data_ptr()))
    s.sync()
    for g, h in ((lam, lam_h), (lam_ac, lam_ac_h)):
        assert np.abs(g.cpu().numpy() - h).max() <= 1e-13 * np.abs(h).max()
    s.close()


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("tile", [64, 128])
def test_ensemble_tubes_by_tile_count(tile, extra):
    """1-D ensembles of 65,536 / tile tiles (general fluxes) and of one more
    (bounded ones), a member beyond the bounded range among them."""
    tc, nt = tile - 1, 65536 // tile
    members = []
    for nx in ((nt - 12) // 2 * tc, 4 * tc, (nt - 12) // 2 * tc, 7 * tc + 5 + extra * tc):
        cfg, uh, um, _ = problems.brio_wu(nx)
        members.append((cfg, uh, um))
    cfg, uh, um = members[1]
    big = um * 2.0 ** 104
    big[5:8] = um[5:8] * 2.0 ** 52
    members[1] = cfg.replace(col=cfg.col * 2.0 ** -104), uh * 2.0 ** 104, big
    e = Ensemble(members, tend=1.0e30, max_steps=3, tile=tile)
    e.set_mode("lockstep")
    e.run()
    for m, (cfg, uh, um) in enumerate(members):
        o = Oracle(cfg, uh, um, None)
        o.run(nsteps=3)
        for g, w in zip(e.state(m), o.state()):
            assert np.array_equal(interior(g, cfg), interior(w, cfg))
    e.close()


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("flow", ["orszag_tang", "kelvin_helmholtz"])
def test_default_tile_of_large_grids(flow, extra):
    """8192 tiles of 16x15 (those) and more (16x7), the last column partial."""
    nx, ny = 52, 15 * 2048 + extra
    cfg, uh, um, _ = cut(flow, nx, 64)
    rows = np.arange(ny + 4) % 64 + 2
    cfg = cfg.replace(ny=ny, ymax=cfg.ymin + ny * cfg.dy)
    same_as_oracle(cfg, uh[:, rows].copy(), um[:, rows].copy(), None, nsteps=2)
