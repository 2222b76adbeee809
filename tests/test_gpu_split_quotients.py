"""The quotients of the Steger-Warming split flux are divisions, rounded once:
of a gas at rest between first-order faces (rows of three nodes) with a metric
of a power of two, the mass and energy fluxes are products and quotients
only, so plain FP64 arithmetic gives the same bits (tolerance 0; the metrics
across the rows are 2^-200, and what they add is lost in rounding)."""
import numpy as np
import pytest

from aerocfd_amd import FlowConfig, cases
from aerocfd_amd import solver as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 64, 5000])
def test_at_rest(rows):
    print("test_at_rest", rows, flush=True)
    g = 1.4
    rng = np.random.default_rng(rows)
    shp = (rows + 2, 3, 3)
    zero = np.zeros(shp)
    rho, p = 1.0 + rng.random(shp), 1.0 + rng.random(shp)
    q = cases.conservative(rho, zero, zero, zero, p)
    mx = 2.0 ** rng.integers(-2, 3, shp)
    dx = np.zeros(shp + (9,))
    dx[..., 0] = mx
    dx[..., 4] = dx[..., 8] = 2.0 ** -200
    r = np.array([0, 2, 0, 2, 0, rows + 1, 0, 2, 0, 2, 0, rows + 1, 1, 1, 1, 1, 1, rows], np.int32)
    got = S.inviscid_flux_1(FlowConfig(ma=0.5, inviscid_scheme=1), r, q, dx, np.ones(shp))[1:-1, 1, 1]

    c = np.sqrt(g * ((g - 1.0) * q[..., 4]) * (1.0 / rho))
    h, s = c * c / (g - 1.0), rho / (2.0 * g)
    mass, energy = s * (mx * c), s * (mx * c * h)  # to the right; to the left the negatives
    for x, f in ((0, mass), (4, energy)):
        face = f[1:-1, 1, :-1] - f[1:-1, 1, 1:]
        want = -(face[:, 1] - face[:, 0])
        assert np.array_equal(got[:, x], want), (x, (got[:, x] != want).sum(), np.abs(got[:, x] - want).max())
