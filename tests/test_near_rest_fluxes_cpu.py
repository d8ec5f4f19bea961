"""The bounded HLLC flux of faces near rest, where the contact speed lies in
the band (0, 5e-11) that its switch passes through (host build, beside the
general flux): covered, and the same values."""
import ctypes

import numpy as np
import pytest

from tests.test_bounded_fluxes_cpu import N, _p, _states, rc  # noqa: F401  (rc: fixture)


@pytest.mark.parametrize("speed", [0.0, 1e-300, 1e-20, 1e-16, 1e-13, 1e-11, 1e-10, 1e-9])
@pytest.mark.parametrize("kind", ["equal", "close", "random"])
def test_faces_near_rest(rc, kind, speed):  # noqa: F811
    l, q = _states(kind)
    r = np.random.default_rng(3)
    l[:, 1], q[:, 1] = speed * r.standard_normal((2, N))
    if kind != "random":  # the same density and pressure on both sides
        q[:, [0, 4]] = l[:, [0, 4]]
    gen, bnd = np.empty((N, 9)), np.empty((N, 9))
    cov = rc.rc_hllc(_p(l), _p(q), ctypes.c_double(5.0 / 3.0), ctypes.c_long(N), _p(gen), _p(bnd))
    assert np.array_equal(gen, bnd)
    assert cov == N

