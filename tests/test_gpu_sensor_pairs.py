"""The shock sensor's kernels take two nodes of a row per thread and cut the
rows into pieces: the flags against the checker's, and whole steps (which form
the gradients on the way) against the stage pieces, at the sizes where a piece
or a pair ends (even and odd rows, one node more and fewer than whole pieces,
boxes all of whose windows meet an end), for every kind of end.  Exact: flags
are bits, and both sides of the second comparison round alike."""
import pytest

from astr_gpu_amd.solver import UDF_RIEMANN2D
from test_gpu_upwind import np, run_both
from test_gpu_upwind_stage import test_steps_equal_pieces as steps_equal_pieces

pytestmark = pytest.mark.gpu

SIZES = [(16, 16, 0), (17, 19, 0), (126, 18, 0), (127, 17, 0), (128, 16, 0), (255, 21, 0),
         (16, 17, 18), (19, 16, 16), (33, 18, 17)]


@pytest.mark.parametrize("npdc", [(3, 3, 3), (1, 2, 3), (2, 1, 1), (4, 3, 2), (3, 4, 4)])
@pytest.mark.parametrize("dims", SIZES)
def test_flags_match_checker(dims, npdc):
    if dims[2] == 0:
        npdc = npdc[:2] + (3,)
    print(f"case sensor {dims} {npdc}", flush=True)
    flagged = 0
    for shkcrt in (0.01, 0.2):
        _, ref, lsh = run_both(dims, npdc, 3, True, shkcrt=shkcrt)
        assert np.array_equal(lsh, ref["lshock"])
        flagged += int(lsh.sum())
    assert flagged > 0


@pytest.mark.parametrize("dims", [(126, 16, 0), (127, 18, 0), (128, 17, 0)])
def test_steps_at_the_pieces_ends(dims):
    steps_equal_pieces((dims, (4, 4, 3), 3, 1, 1, (0, 0, 0, 0, 1, 1), UDF_RIEMANN2D))
    steps_equal_pieces((dims, (3, 4, 3), 3, 1, 1, (1, 1, 60, 50, 1, 1), 0))
