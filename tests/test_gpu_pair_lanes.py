"""The pair list's forms by size and stencil (8 or 4 lanes a bead, 9 or 27
cells), on either side of 200,000 beads and with folded axes of one layer,
against the FP64 oracle as test_gpu_pair_list's."""
import pytest

from test_gpu_pair_list import test_pair_list_against_oracle as against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,W,n,wca,activity", [
    ((23, 40, 1), 60, 11, False, 0.3), ((2, 31, 1), 9, 7, False, 0.3), ((1, 9, 1), 7, 5, True, 0.3),
    ((40, 37, 1), 90, 13, True, 0.3), ((520, 510, 1), 20_000, 10, True, 0.3), ((520, 510, 1), 20_001, 10, True, 0.3),
    ((520, 510, 1), 20_001, 10, False, 0.3), ((66, 64, 62), 20_001, 10, True, 0.0), ((66, 64, 62), 20_001, 10, False, 0.3)])
def test_lanes_against_oracle(nwlib, grid, W, n, wca, activity):
    against_oracle(nwlib, grid, W, n, wca, activity)
