"""Whole upwind steps with statistics: the first stage of every step, the later
ones of a call too, stores the gradients for them and forms the shock sensor
from the stored ones.  Statistics, state, residual, gradients and shock flags
against the stage pieces with statcal after the first rhscal, bit for bit (the
same kernels on the same values).  A two-dimensional box has no statistics: the
steps refuse to form them."""
import numpy as np
import pytest

import astr_gpu_amd as ag
from test_gpu_upwind import quadrant_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,conv,explicit,filt", [
    ((16, 18, 17), 1, 1, 0), ((33, 17, 20), 1, 1, 1), ((24, 20, 18), 1, 0, 0), ((20, 16, 18), 2, 1, 0)])
def test_statistics_of_steps_equal_pieces(dims, conv, explicit, filt):
    print(f"case upwind statistics {dims} {conv} {explicit} {filt}", flush=True)
    p = ag.default_params(dims, convection=conv, deriv_explicit=explicit, recon_schem=3,
                          lchardecomp=1, lfilter=filt, diffterm=0, mach=1.0)
    st = quadrant_state(dims)
    n, dt = 3, 2e-4
    out = []
    for whole in (True, False):
        s = ag.AstrSolver(p)
        s.upload_geom(*ag.box_metrics(p, lengths=(1.0, 1.0, 1.0)))
        s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
        if whole:
            stats = s.steploop(n, dt, stats=True)
        else:
            stats = np.zeros((n, 3))
            for k in range(n):
                for stage in (1, 2, 3):
                    if filt:
                        s.filterq()
                    s.qswap()
                    s.rhscal()
                    if stage == 1:
                        stats[k] = s.statcal()
                    s.rk3_update(stage, dt)
        out.append({**s.download_state(), **s.download_rhs(), "stats": stats,
                    "shock": s.download_shock()})
        s.close()
    assert np.all(out[0]["stats"][0, :2] > 0.0)
    for nm in out[0]:
        # (the filter across these shocks leaves negative temperatures, whose
        # viscosity is no number: both sides' alike)
        assert np.array_equal(out[0][nm], out[1][nm], equal_nan=True), nm
        assert filt or np.all(np.isfinite(out[0][nm])), nm


def test_two_dimensional_steps_refuse_statistics():
    p = ag.default_params((20, 18, 0), convection=1, deriv_explicit=1, lfilter=0, diffterm=0, mach=1.0)
    s = ag.AstrSolver(p)
    s.upload_geom(*ag.box_metrics(p, lengths=(1.0, 1.0, 1.0)))
    st = quadrant_state((20, 18, 0))
    s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
    with pytest.raises(ag.AstrError):
        s.steploop(2, 2e-4, stats=True)
    s.close()
