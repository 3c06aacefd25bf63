"""A batch set right behind another takes nothing over from it: a passive WCA
batch behind one with the extensile term, or with soft spheres, needs no
sorted tangents, can be differentiated and steps bit for bit as by itself."""
import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, lattice_system_2d

pytestmark = pytest.mark.gpu


def batch(lib, activity=0.0, wca=True):
    R, n = 3, 9
    reps, pos, vel = (abi.NWReplicaParams * R)(), [], []
    for r in range(R):
        p, a, b = lattice_system_2d(40 + 7 * r, n, 34, np.random.default_rng(r))
        p.activity = activity
        reps[r].params, reps[r].seed = p, 9 + r
        reps[r].ext = ext_params(pairPotential=abi.NW_PAIR_WCA if wca else abi.NW_PAIR_REF_DEM,
                                 bondedMode=abi.NW_BONDED_CHAIN, driveForce=3.0, stencil=abi.NW_STENCIL_2D)
        pos.append(a)
        vel.append(b)
    lib.nwBatchSetReplicas(reps, R)
    return [np.concatenate(x) for x in (pos, vel)]


def steps(lib, pos, vel):
    N = len(pos)
    d = [DeviceArray.from_numpy(lib, x) for x in (pos, vel, *[np.zeros_like(pos)] * 3)]
    w = [DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)]
    lib.nwBatchMdStep(*[x.p for x in d], w[0].p, w[1].p, None, None, 1e-3, 3, 0)
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    lib.nwBatchAdjointForward(*[x.p for x in d], 1e-3, 0, None, 3, 2)
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    return [x.download(np.uint32, (N, 4)) for x in d]


@pytest.mark.parametrize("before", [dict(activity=2.0), dict(wca=False)])
def test_passive_batch_behind_another(nwlib, before):
    lib = nwlib
    try:
        lib.nwBatchSetReplicas(None, 0)
        alone = steps(lib, *batch(lib))
        lib.nwBatchSetReplicas(None, 0)
        batch(lib, **before)
        behind = steps(lib, *batch(lib))
    finally:
        lib.nwBatchSetReplicas(None, 0)
    for name, a, b in zip(("pos", "vel", "force", "forceOld", "tangent"), alone, behind):
        assert np.array_equal(a, b), name
