"""filterq writes the nodes 0..n only, on bounded axes too: the last y and z
tiles also stage, and store back as they were, the x columns after node n up to
the end of its 128-byte line, and a wavefront solves two lines at once, so with
an odd number of lines in the last tile (n even) one of those columns sits in a
solve.  Every cell outside the nodes, the columns on the rows of the closures
among them, comes back bit for bit, at every number of rows per lane whose
closure rows pass through LDS (1, 2, 3) and the one after."""
import numpy as np
import pytest

import astr_gpu_amd as ag

pytestmark = pytest.mark.gpu
HM = 5


@pytest.mark.parametrize("npdc", [(3, 4, 3), (3, 3, 4), (4, 4, 4), (4, 3, 3)])
@pytest.mark.parametrize("dims", [(16, 17, 24), (18, 40, 26), (32, 57, 58), (40, 89, 70),
                                  (17, 25, 90), (30, 90, 16)])
def test_cells_outside_the_nodes(dims, npdc):
    print(f"case filterq keeps dims={dims} npdc={npdc}", flush=True)
    p = ag.default_params(dims, npdci=npdc[0], npdcj=npdc[1], npdck=npdc[2])
    s = ag.AstrSolver(p)
    s.upload_geom(*ag.box_metrics(p))
    rng = np.random.default_rng(4)
    shp = ag.haloed_shape(p)
    q = np.asfortranarray(1.0 + 0.1 * rng.standard_normal(shp + (5,)))
    one = np.asfortranarray(np.ones(shp))
    s.upload_state(q, one, np.asfortranarray(np.zeros(shp + (3,))), one, one)
    s.filterq()
    out = s.download_state()["q"]
    s.close()
    inside = np.zeros(shp, dtype=bool)
    inside[HM:HM + dims[0] + 1, HM:HM + dims[1] + 1, HM:HM + dims[2] + 1] = True
    for m in range(5):
        assert np.array_equal(out[..., m][~inside], q[..., m][~inside]), m
        assert not np.array_equal(out[..., m][inside], q[..., m][inside]), m
