"""The y and z gradients of a stage, one launch where both axes take the same
rows per lane (25 | 26, 57 | 58 and 89 | 90 cells are the last and first
lengths of 1, 2, 3 and 4) and two where they do not, against the field
derivative of each velocity component and the temperature times the metric.
Tolerance: a right-hand side row is 4 products of values up to max|f| with
coefficients that sum to 2 in magnitude, wrong by 5 eps of that, and the
system's inverse is at most 1 / (1 - 2/3) = 3 in the maximum norm: 30 eps
max|f| on each side, times the metric, and 2 eps of the result for that
product."""
import numpy as np
import pytest

import astr_gpu_amd as ag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(16, 16, 16), (18, 25, 17), (17, 26, 57), (20, 58, 89), (16, 90, 91),
                                  (19, 25, 26), (16, 58, 57)])
def test_gradients_match_field_derivatives(dims):
    print(f"case grad yz {dims}", flush=True)
    p = ag.default_params(dims)
    s = ag.AstrSolver(p)
    jac, dxi = ag.box_metrics(p)
    s.upload_geom(jac, dxi)
    st = ag.tgv_state(p)
    rng = np.random.default_rng(11)
    st["q"] = np.asfortranarray(st["q"] * (1.0 + 0.01 * rng.random(st["q"].shape)))
    s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
    s.qswap()
    s.rhscal()
    h, r = s.download_state(), s.download_rhs()
    eps = np.finfo(float).eps
    for d in (1, 2):
        xi = ag.interior(dxi[..., d, d], p)
        for f, g in [(h["vel"][..., m], r["dvel"][..., m, d]) for m in range(3)] + [(h["tmp"], r["dtmp"][..., d])]:
            ref = s.central(d + 1, np.asfortranarray(f)) * xi
            tol = 60 * eps * np.max(np.abs(f)) * np.max(xi) + 2 * eps * np.max(np.abs(ref))
            assert np.max(np.abs(g - ref)) <= tol, d
    s.close()
