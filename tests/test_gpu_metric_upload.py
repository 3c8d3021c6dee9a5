"""The metric fields of a grid with general metrics are allocated by the first
upload and filled from the context's stream: what that upload leaves is what a
second one, into the same fields, leaves.  Seen through the gradients and the
right-hand side of one stage, bit for bit, on several fresh contexts."""
import numpy as np
import pytest

import astr_gpu_amd as ag
from test_gpu_curvilinear import state, wavy_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(20, 17, 16), (96, 80, 72)])
def test_first_upload_equals_second(dims):
    print(f"case metric upload {dims}", flush=True)
    X, Y, Z, jac, dxi = wavy_grid(dims)
    st = state(X, Y, Z)
    p = ag.default_params(dims)
    for _ in range(3):
        s = ag.AstrSolver(p)
        s.upload_state(st["q"], st["rho"], st["vel"], st["prs"], st["tmp"])
        out = []
        for _ in range(2):
            s.upload_geom(jac, dxi)
            s.rhscal()
            out.append(s.download_rhs())
        s.close()
        for nm in out[0]:
            assert np.all(np.isfinite(out[0][nm])) and np.any(out[0][nm] != 0.0)
            assert np.array_equal(out[0][nm], out[1][nm]), nm
