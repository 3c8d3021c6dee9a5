"""k_row_flux (the x gradient, the fluxes G and the x flux derivative of one
row) at the row lengths where it can go wrong: the last length of a
rows-per-lane count and the first of the next (25/26, 57/58, 89/90), rows
that end a 128-byte line (31, 47) or start one (32, 48), the shortest row,
and a bounded x axis.  Tolerance: the 1e-10 of whole steps against the
checker (a few steps of rounding, ~1e-13, leave three orders of margin)."""
import numpy as np
import pytest

import astr_gpu_amd as ag
import pyoracle
from test_gpu_parity import compare_state

pytestmark = pytest.mark.gpu


def pair(dims, npdci=3):
    npdc = (npdci, 3, 3)
    ob = pyoracle.OracleBox(dims, variant=0, npdc=npdc)
    ob.init_tgv()
    st = ob.state_haloed()
    p = ag.default_params(dims, npdci=npdci)
    s = ag.AstrSolver(p)
    s.upload_geom(*ag.box_metrics(p))
    s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
    return ob, s, p, st


@pytest.mark.parametrize("nx,npdci", [(16, 3), (25, 3), (26, 3), (31, 3), (32, 3), (47, 3), (48, 3),
                                      (57, 3), (58, 3), (89, 3), (90, 3), (25, 4), (58, 4)])
def test_rows_match_checker(nx, npdci):
    dims = (nx, 18, 16)
    print(f"case rows dims={dims} npdci={npdci}", flush=True)
    ob, s, p, _ = pair(dims, npdci)
    for n in range(2):
        so = ob.step(0.002, stats=True)
        sg = s.time_integration_rk(0.002, stats=True)
        for a, b in zip(sg, so):
            assert abs(a - b) <= 1e-10 * abs(b), (n, sg, so)
    compare_state(ob, s, p, 1e-10, halo_faces=True, vector_scale=True)
    s.close()
    ob.close()


def test_gradients_after_steps():
    """The gradients that statcal and download_rhs read after whole steps are
    those of the last stage, as when the stages run call by call."""
    dims, dt = (41, 20, 18), 0.002
    ob, s1, p, st = pair(dims)
    ob.close()
    s2 = ag.AstrSolver(p)
    s2.upload_geom(*ag.box_metrics(p))
    s2.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
    s1.steploop(2, dt)
    for _ in range(2):
        for stage in (1, 2, 3):
            s2.filterq()
            s2.qswap()
            s2.rhscal()
            s2.rk3_update(stage, dt)
    a, b = s1.download_rhs(), s2.download_rhs()
    for nm in ("dvel", "dtmp"):
        assert np.max(np.abs(a[nm] - b[nm])) <= 1e-12 * np.max(np.abs(b[nm])), nm
    for x, y in zip(s1.statcal(), s2.statcal()):
        assert abs(x - y) <= 1e-12 * abs(y)
    s1.close()
    s2.close()
