"""The bounded HLLC flux where the contact speed is not finite (host build,
beside the general flux)."""
import ctypes

import numpy as np

from tests.test_bounded_fluxes_cpu import N, _p, rc  # noqa: F401  (rc: fixture)


def test_contact_speeds_that_are_not_finite(rc):  # noqa: F811
    """The divisor of the contact speed passes through zero in supersonic flow
    (1.03 multiplies signed wave speeds: at densities 1 and 2 near 103 sound
    speeds): whatever the flux is there, the two functions agree."""
    l, q = np.zeros((N, 9)), np.zeros((N, 9))
    l[:, 0], l[:, 4] = 1.0, 0.6
    q[:, 0], q[:, 4] = 2.0, 1.2
    v = -np.sqrt(5.0 / 3.0 * 0.6) * (3.09 / 0.03)
    l[:, 1] = q[:, 1] = v + (np.arange(N) - N // 2) * np.spacing(v)
    l[:, 2], q[:, 3] = 0.5, -0.25
    gen, bnd = np.empty((N, 9)), np.empty((N, 9))
    cov = rc.rc_hllc(_p(l), _p(q), ctypes.c_double(5.0 / 3.0), ctypes.c_long(N), _p(gen), _p(bnd))
    assert np.array_equal(gen, bnd, equal_nan=True)
    assert cov < N
