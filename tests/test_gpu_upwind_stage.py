"""Whole upwind steps, whose inner stages form the shock sensor without
storing the gradients, refresh the primitives of a 2-D box on its edges only
and let the first axis set qrhs, against the stage pieces (boucon, qswap,
rhscal, rk3_update), which store and refresh everything: the state with its
halos, the residual, the gradients and the shock flags, bit for bit.  The
sizes have boxes whose sensor windows all meet an end (16), and blocks and
tiles that end inside the box."""
import numpy as np
import pytest

import astr_gpu_amd as ag
from astr_gpu_amd.solver import UDF_RIEMANN2D

pytestmark = pytest.mark.gpu

CASES = [
    # dims, npdc, recon, convection, lchardecomp, bctype, udf
    ((16, 16, 0), (4, 4, 3), 3, 1, 1, (0, 0, 0, 0, 1, 1), UDF_RIEMANN2D),
    ((47, 33, 0), (4, 4, 3), 3, 1, 1, (0, 0, 0, 0, 1, 1), UDF_RIEMANN2D),
    ((40, 273, 0), (4, 4, 3), 5, 1, 1, (50, 23, 42, 23, 1, 1), 0),
    ((270, 20, 0), (3, 4, 3), 2, 1, 1, (1, 1, 60, 50, 1, 1), 0),
    ((33, 30, 0), (3, 3, 3), -1, 1, 0, (1,) * 6, 0),
    ((30, 25, 0), (4, 3, 3), 3, 2, 1, (1,) * 6, 0),
    ((16, 18, 17), (3, 3, 3), 3, 1, 1, (1,) * 6, 0),
    ((33, 17, 20), (3, 3, 3), 5, 1, 1, (1,) * 6, 0),
    ((20, 16, 18), (3, 3, 3), 0, 2, 1, (1,) * 6, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-{c[2]}-{c[3]}" for c in CASES])
def test_steps_equal_pieces(case):
    dims, npdc, recon, conv, lchar, bctype, udf = case
    print(f"case upwind stage {case}", flush=True)
    p = ag.default_params(dims, npdci=npdc[0], npdcj=npdc[1], npdck=npdc[2], convection=conv,
                          deriv_explicit=1, recon_schem=recon, lchardecomp=lchar, lfilter=0,
                          diffterm=0, mach=1.0)
    st = ag.riemann2d_state(p)
    # primitives that q does not give: a call takes the state as it is
    rng = np.random.default_rng(7)
    st["prs"] = np.asfortranarray(st["prs"] * (1.0 + 1e-3 * rng.standard_normal(st["prs"].shape)))
    out = []
    n, dt = 3, 2e-4
    for whole in (True, False):
        s = ag.AstrSolver(p)
        s.upload_geom(*ag.box_metrics(p, lengths=(1.0, 1.0, 1.0)))
        s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
        s.set_lengths(1.0, 1.0, 1.0)
        s.set_bc(bctype, udf)
        if whole:
            s.steploop(n, dt)
        else:
            for k in range(n):
                s.time = k * dt
                for stage in (1, 2, 3):
                    s.boucon()
                    s.qswap()
                    s.rhscal()
                    s.rk3_update(stage, dt)
        d = {**s.download_state(), **s.download_rhs()}
        d["shock"] = s.download_shock()
        out.append(d)
        s.close()
    for nm in out[0]:
        assert np.array_equal(out[0][nm], out[1][nm], equal_nan=True), nm
