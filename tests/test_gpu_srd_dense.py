"""The collision's cells of dense solvents, on both sides of each line of the
sort's second level (nw_rules.hpp: its network, its placement): the order of a
stable sort by cell exactly, the cells' mean velocities against sums in FP64
(a mean of some tens of FP32 terms: 1e-5 of the speeds)."""
import ctypes

import numpy as np
import pytest

from nwamd.abi import DeviceArray
from nwtest import ext_params, sim_params, solvent_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per,L", [(8, 64), (12, 64), (13, 63), (20, 64), (21, 63), (45, 64), (130, 33),
                                   (8, 400), (9, 560), (11, 560), (20, 420), (30, 420)])
@pytest.mark.parametrize("ordered", [False, True])
def test_dense_cells(nwlib, per, L, ordered):
    lib, rng = nwlib, np.random.default_rng([per, L, int(ordered)])
    Ns = per * L * L + 1 if per in (12, 20) else per * L * L
    p = sim_params(grid=(L, L, 1), cell=1.0, W=0, n=3)
    s = solvent_params(p, (L, L, 1), (1.0, 1.0, 1.0), alpha=1.0, kbT=0.3, offset=(0.0, 0.0, 0.0), ns=Ns)
    pos, vel = np.zeros((Ns, 4), np.float32), np.zeros((Ns, 4), np.float32)
    pos[:, :2] = (rng.random((Ns, 2)) - 0.5) * L * 0.999
    if ordered:
        c = np.floor(pos[:, 1] + L / 2) * L + np.floor(pos[:, 0] + L / 2)
        pos = pos[np.argsort(c, kind="stable")]
    pos[:, 2] = p.origin.z + 0.5
    vel[:, :2] = rng.normal(0, 1, (Ns, 2))
    vel[:, 3] = 1.0
    lib.setParameters(ctypes.byref(p))
    lib.setSolventParameters(ctypes.byref(s))
    lib.nwSetExtParameters(ctypes.byref(ext_params()))
    P, V = DeviceArray.from_numpy(lib, pos), DeviceArray.from_numpy(lib, vel)
    h, i, com = DeviceArray(lib, 4 * Ns), DeviceArray(lib, 4 * Ns), DeviceArray(lib, 16 * L * L)
    lib.nwFusedSrdStep(P.p, V.p, com.p, h.p, i.p, 0.01, 0, Ns, 0)
    hash_, ids = h.download(np.uint32, (Ns,)), i.download(np.uint32, (Ns,))
    assert np.array_equal(ids, np.argsort(hash_, kind="stable"))
    n = np.bincount(hash_, minlength=L * L)
    mean = np.stack([np.bincount(hash_, vel[:, k].astype(np.float64), L * L) for k in range(3)], 1)
    mean /= np.maximum(n, 1)[:, None]
    assert np.abs(com.download(np.float32, (L * L, 4))[:, :3] - mean).max() < 5e-5
