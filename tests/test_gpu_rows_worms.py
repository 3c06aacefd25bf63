"""The one-launch cell order and pair pass finds its beads by the rows of cells
that every worm spans: rounds of worms (more than 8,192), long worms, more
rows a workgroup, worms across the box's y edge (which every workgroup lists,
past its list), against the sort and the pair kernel.  Bit for bit."""
import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import NWTuning
from nwtest import ext_params, random_forces, random_worms, sim_params
from test_gpu_rows import lib, step  # noqa: F401 (lib is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,W,n,how", [
    ((130, 121), 8192, 1, ""), ((130, 121), 8193, 2, ""), ((200, 190), 24576, 1, ""), ((500, 480), 2000, 64, ""),
    ((420, 600), 9000, 20, ""), ((60, 700), 2500, 9, ""), ((80, 80), 5000, 1, "few rows"), ((90, 80), 5000, 2, "edge")])
def test_worm_rows_equal_sort_and_pairs(lib, grid, W, n, how):  # noqa: F811
    rng = np.random.default_rng([*grid, W, n])
    p = sim_params(grid=(*grid, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
    e = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                   stencil=abi.NW_STENCIL_2D)
    pos, vel, tan = random_worms(p, rng, twod=True)
    if how == "few rows":
        pos[:, 1] *= np.float32(0.015)
    if how == "edge":
        pos[0::2, 1], pos[1::2, 1] = p.origin.y + p.boxSize.y - 0.1, p.origin.y + 0.3
        pos[1::2, 0] = pos[0::2, 0]
    f = random_forces(rng, W * n, 0.5)
    state = (pos, vel, f, f[::-1].copy(), tan)
    a = step(lib, p, e, state, NWTuning(), 0)
    b = step(lib, p, e, state, NWTuning(mdMembers=512), 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "hash", "ids", "sortedPos"), a, b):
        assert np.array_equal(x, y), (name, int((x != y).sum()))
