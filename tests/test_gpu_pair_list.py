"""The pair pass over any stencil (nw_pairs.hip), through collideFilaments and
through a fused step over several layers, against the FP64 oracle: grids whose
axes fold the 27 offsets, odd bead counts (the last workgroup is ragged), and
cells so full that a bead's candidates pass the list a group of lanes keeps."""
import ctypes

import numpy as np
import pytest

import orc
from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, force_tol_check, random_forces, random_worms, sim_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,W,n,wca,activity", [
    ((3, 3, 3), 13, 31, False, 0.2),    # ~130 candidates a bead: several rounds of the list
    ((3, 3, 3), 1, 1, False, 0.2),      # a single bead
    ((4, 3, 5), 7, 9, False, 0.0),      # 63 beads, one ragged workgroup
    ((2, 5, 3), 11, 10, False, 0.3),    # x folds: weights 1 and 2
    ((1, 2, 4), 9, 7, False, 0.3),      # x and y fold: weights up to 6
    ((1, 1, 1), 6, 11, False, 0.3),     # one cell, weight 27, more than a list of itself
    ((9, 7, 11), 60, 10, True, 0.0),    # WCA over several layers
    ((9, 7, 11), 60, 10, True, 0.3),
    ((2, 8, 6), 8, 10, True, 0.0),
])
def test_pair_list_against_oracle(nwlib, grid, W, n, wca, activity):
    rng = np.random.default_rng([*grid, W, n, int(wca), int(10 * activity)])
    lib = nwlib
    p = sim_params(grid=grid, cell=1.2 if wca else 1.0, W=W, n=n, bondSpringL=0.8 if wca else 0.4, activity=activity)
    e = ext_params(pairPotential=abi.NW_PAIR_WCA if wca else abi.NW_PAIR_REF_DEM, stencil=abi.NW_STENCIL_REF27)
    pos, vel, tan = random_worms(p, rng)
    force = random_forces(rng, W * n, 0.1)
    h, i = orc.calc_hash(p, None, pos)
    h, i = orc.sort_pairs(h, i)
    cs, ce, sp, sv, st = orc.reorder(h, i, pos, vel, tan, p.numCells)
    ref = orc.collide_filaments(p, e, sp, sv, st, i, cs, ce, force)
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    d = [DeviceArray.from_numpy(lib, a) for a in (force, sp, sv, st, i, cs, ce)]
    lib.collideFilaments(*[x.p for x in d], W * n, p.numCells)
    force_tol_check(d[0].download(np.float32, (W * n, 4)), ref, name="collideFilaments")
    # a fused step of length 0 from zero forces: the pair forces alone, on the same positions
    zero = np.zeros_like(pos)
    e.bondedMode = abi.NW_BONDED_REF
    p.bondBendingK = 0.0
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    a = [DeviceArray.from_numpy(lib, x) for x in (pos, vel, zero, zero, tan)]
    hd, idd = DeviceArray(lib, 4 * W * n), DeviceArray(lib, 4 * W * n)
    s = [DeviceArray(lib, 16 * W * n) for _ in range(3)]
    lib.nwFusedMdStep(*[x.p for x in a], hd.p, idd.p, *[x.p for x in s], 0.0, 0.0, 0.0, 0, W)
    tan2 = a[4].download(np.float32, (W * n, 4))
    assert np.array_equal(idd.download(np.uint32, (W * n,)), i)
    ref = orc.collide_filaments(p, e, sp, sv, tan2[i], i, cs, ce, zero)
    force_tol_check(a[2].download(np.float32, (W * n, 4)), ref, name="fused step")
