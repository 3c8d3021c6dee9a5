"""k_row_flux at the long rows, whose instances run with more registers and
fewer wavefronts: the last length of a rows-per-lane count and the first of the
next (313/314, 441/442), and the longest a line takes (505), against the checker
as the shorter rows."""
import pytest

from test_gpu_row_flux import test_rows_match_checker as rows_match_checker

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,npdci", [(313, 3), (314, 3), (441, 3), (442, 4), (505, 3), (505, 4)])
def test_long_rows_match_checker(nx, npdci):
    rows_match_checker(nx, npdci)
