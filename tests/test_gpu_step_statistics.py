"""The statistics a whole step forms with the fluxes keep their partial sums in
double-double from node to node of a row: a row of 504 cells whose first 63
nodes have u = 1 and whose other 441 u^2 = 0.945 * 2^-53, each of which, added
to a sum of 1 in plain double, is lost.  With rho = 1, v = w = 0 every term of
the kinetic energy is exact, so the mean is known exactly; the result may be
off by the final rounding of the sum and of its division, one unit of 2^-52
each at most half, and the halving is exact: 1.5 * 2^-52 leaves half a unit."""
from fractions import Fraction

import numpy as np
import pytest

import astr_gpu_amd as ag

pytestmark = pytest.mark.gpu
HM = 5


@pytest.mark.parametrize("nx", [504, 300, 130])
def test_kinetic_energy_sum_of_a_row(nx):
    dims = (nx, 17, 16)
    print(f"case step statistics {dims}", flush=True)
    p = ag.default_params(dims, lfilter=0)
    s = ag.AstrSolver(p)
    s.upload_geom(*ag.box_metrics(p))
    shp = ag.haloed_shape(p)
    small = 1.375 * 2.0 ** -27
    u = np.full(shp, small, order="F")
    u[HM + 1:HM + 64] = 1.0
    one = np.asfortranarray(np.ones(shp))
    vel = np.zeros(shp + (3,), order="F")
    vel[..., 0] = u
    prs = np.asfortranarray(one / (p.gamma * p.mach ** 2))
    q = np.zeros(shp + (5,), order="F")
    q[..., 0] = 1.0
    q[..., 1] = u
    q[..., 4] = prs / (p.gamma - 1.0) + 0.5 * u * u
    s.upload_state(q, one, vel, prs, one)
    ke = s.time_integration_rk(1e-6, stats=True)[0]
    s.close()
    exact = (63 + (nx - 63) * Fraction(small) ** 2) / (2 * nx)
    err = abs(Fraction(ke) - exact) / exact * 2 ** 52
    print(f"  {float(err):.2f} units of 2^-52")
    assert err <= Fraction(3, 2)
