"""The compact filter on short lines, whose closure rows are taken one per
lane, against the checker line by line, for every kind of end, at the lengths
where the rows per lane change (1, 2, 3 | 4) and on either side of them.
Tolerance: a right-hand side row is a dot product of at most 11 terms whose
coefficients sum to at most 2 in magnitude, wrong by at most 12 eps times
that; the system's inverse is at most 1 / (1 - 2 0.49) = 50 in the maximum
norm: 50 * 12 * 2 eps = 2.7e-13 of the line's largest value."""
import numpy as np
import pytest

import astr_gpu_amd as ag
import pyoracle
from test_gpu_parity import lines_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntype", [1, 2, 3, 4])
@pytest.mark.parametrize("dims", [(16, 17, 24), (25, 26, 19), (57, 16, 58), (20, 57, 89), (89, 90, 16)])
def test_closure_rows(dims, ntype):
    print(f"case filter closures {dims} {ntype}", flush=True)
    p = ag.default_params(dims, npdci=ntype, npdcj=ntype, npdck=ntype)
    s = ag.AstrSolver(p)
    rng = np.random.default_rng(ntype)
    f = np.asfortranarray(rng.standard_normal(ag.haloed_shape(p)))
    for d in (1, 2, 3):
        ff = s.compact_filter(d, f)
        ref = lines_ref(lambda ln: pyoracle.compact_filter(ntype, ln), f, d)
        assert np.max(np.abs(ff - ref)) <= 2.7e-13 * np.max(np.abs(f))
    s.close()
