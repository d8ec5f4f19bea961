"""The fluxes and face states for bounded states against the general ones,
value for value (host build of pip_riemann.h and pip_phys.h): every HLLD and
HLLC region, equal sides, fields and velocities that are zero or tiny, wide
ratios.  The device forms share the algebra; their quotients and roots are the
sequences test_gpu_arith checks, and the parity tests run them in the kernels."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
N = 200_000


@pytest.fixture(scope="module")
def rc(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rc") / "riemanncheck.so")
    subprocess.check_call(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-shared", "-fPIC",
                           "-I", os.path.join(HERE, "..", "pip_amd", "csrc"), "-o", so,
                           os.path.join(HERE, "riemanncheck.cpp")])
    lib = ctypes.CDLL(so)
    lib.rc_hlld.restype = lib.rc_hllc.restype = ctypes.c_long
    return lib


def _p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _states(kind):
    r = np.random.default_rng(len(kind))
    wide = kind in ("random", "wide", "normal field")
    amp = np.exp(r.uniform(-4, 4, (N, 1))) if wide else 1.0
    l, q = r.standard_normal((N, 9)) * amp, r.standard_normal((N, 9)) * amp
    pos = np.exp(r.uniform(-8, 8, (N, 4)) if wide else r.uniform(-1, 1, (N, 4)))
    l[:, 0], q[:, 0], l[:, 4], q[:, 4] = pos.T
    if kind == "close":
        q = l * (1.0 + 1e-3 * r.standard_normal((N, 9)))
    elif kind == "equal":
        q = l.copy()
    elif kind == "mirror":
        q = l.copy()
        q[:, 1] = -l[:, 1]
    elif kind == "normal field":
        q[:, 5] = l[:, 5]
    elif kind == "zeros":
        z = r.random((N, 9)) < 0.5
        z[:, [0, 4]] = False
        l[z], q[z] = 0.0, 0.0
    elif kind == "at rest":
        l[:, 1] *= 1e-12
        q[:, 1] *= 1e-12
        q[:, [0, 4]] = l[:, [0, 4]]
    elif kind == "wide":
        l[:, [0, 4]] *= np.exp(r.uniform(-40, 40, (N, 2)))
        q[:, [0, 4]] *= np.exp(r.uniform(-40, 40, (N, 2)))
    return np.ascontiguousarray(l), np.ascontiguousarray(q)


@pytest.mark.parametrize("gm", [5.0 / 3.0, 1.4])
@pytest.mark.parametrize("kind", ["random", "close", "equal", "mirror", "normal field", "zeros", "at rest", "wide"])
def test_fluxes(rc, kind, gm):
    l, q = _states(kind)
    gen, bnd = np.empty((N, 9)), np.empty((N, 9))
    for nv in (8, 9):
        cov = rc.rc_hlld(nv, _p(l), _p(q), ctypes.c_double(gm), ctypes.c_double(1.3), ctypes.c_long(N), _p(gen),
                         _p(bnd))
        assert np.array_equal(gen, bnd, equal_nan=True)
        assert cov > 0.95 * N
    cov = rc.rc_hllc(_p(l), _p(q), ctypes.c_double(gm), ctypes.c_long(N), _p(gen), _p(bnd))
    assert np.array_equal(gen, bnd, equal_nan=True)
    assert cov > 0.4 * N  # at rest, half of the contact speeds lie in the switch band


def test_face_states(rc):
    r = np.random.default_rng(5)
    a = r.standard_normal((N, 4))
    a[::2] = r.integers(-2, 3, (N // 2, 4))  # ties and zero slopes
    gen, bnd = np.empty((N, 2)), np.empty((N, 2))
    rc.rc_states(_p(a), ctypes.c_long(N), _p(gen), _p(bnd))
    assert np.array_equal(gen, bnd)


def test_bounded_cells(rc):
    ok = np.array([1.0, 0.5, -2.0, 0.0, 1e-8, 1.0, -1.0, 0.0, 0.0])
    assert rc.rc_bounded(_p(ok), 9) == 1
    for k in range(9):
        for bad in (np.nan, np.inf, -np.inf, 2.0 ** 100):
            v = ok.copy()
            v[k] = bad
            assert rc.rc_bounded(_p(v), 9) == 0
    for k in (0, 4):
        for bad in (0.0, -1.0, 2.0 ** -100):
            v = ok.copy()
            v[k] = bad
            assert rc.rc_bounded(_p(v), 9) == 0
