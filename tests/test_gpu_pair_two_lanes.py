"""The pair list with two lanes a bead (large systems of one layer) against the
FP64 oracle as test_gpu_pair_list's: every pair term, a ragged last
workgroup, an axis that folds the offsets, and beads whose candidates take
several rounds of the shorter list."""
import pytest

from test_gpu_pair_list import test_pair_list_against_oracle as against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,W,n,wca,activity", [
    ((520, 510, 1), 20_001, 10, True, 0.0), ((520, 510, 1), 15_387, 13, False, 0.0),
    ((2, 90_000, 1), 20_001, 10, False, 0.3),   # x folds: weights 1 and 2
    ((180, 170, 1), 20_001, 10, False, 0.3),    # ~60 candidates a bead
    ((180, 170, 1), 20_001, 10, True, 0.3)])
def test_two_lanes_against_oracle(nwlib, grid, W, n, wca, activity):
    against_oracle(nwlib, grid, W, n, wca, activity)
