"""The Riemann example's four faces set in one launch against the same faces
two at a time (faces 1, 2 then 3, 4, the reference's order): q, the primitives
and the halos, bit for bit, at times before, while and after the shocks pass
the corners (whole steps, which also refresh the rim in that launch, are
compared with the stage pieces in test_gpu_upwind_stage)."""
import numpy as np
import pytest

import astr_gpu_amd as ag
from astr_gpu_amd.solver import UDF_RIEMANN2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("time", [0.0, 0.3, 2.0])
@pytest.mark.parametrize("dims", [(16, 16, 0), (17, 40, 0), (65, 19, 0), (64, 33, 0)])
def test_rim_equals_faces(dims, time):
    print(f"case rim {dims} {time}", flush=True)
    p = ag.default_params(dims, npdci=4, npdcj=4, npdck=3, convection=1, deriv_explicit=1,
                          recon_schem=3, lchardecomp=1, lfilter=0, diffterm=0, mach=1.0)
    st = ag.riemann2d_state(p)
    rng = np.random.default_rng(5)
    for k in ("rho", "vel", "prs"):
        st[k] = np.asfortranarray(st[k] * (1.0 + 0.01 * rng.standard_normal(st[k].shape)))
    out = []
    for sets in (((0, 0, 0, 0, 1, 1),), ((0, 0, 1, 1, 1, 1), (1, 1, 0, 0, 1, 1))):
        s = ag.AstrSolver(p)
        s.upload_geom(*ag.box_metrics(p, lengths=(1.0, 1.0, 1.0)))
        s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
        s.set_lengths(1.0, 1.0, 1.0)
        s.time = time
        for bc in sets:
            s.set_bc(bc, UDF_RIEMANN2D)
            s.boucon()
        out.append(s.download_state())
        s.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
    assert not np.array_equal(out[0]["q"], st["q"])
