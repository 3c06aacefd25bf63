"""nwBatchPolarSpeedGrad (one launch for the batch) against nwPolarSpeedGrad of
each replica alone: the gradients bit for bit (the same FP32 expressions), the
polar speeds to FP64 rounding over at most 10^4 terms, for worms of 1 to 64
beads, several wavefronts a replica, and a replica without tangents."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, random_worms, sim_params

pytestmark = pytest.mark.gpu


def test_batch_equals_each_replica(nwlib):
    lib = nwlib
    rng = np.random.default_rng(3)
    sizes = [(5, 1), (1, 2), (7, 3), (130, 5), (3, 64), (41, 33), (600, 12)]
    reps, pos, vel = (abi.NWReplicaParams * len(sizes))(), [], []
    for r, (W, n) in enumerate(sizes):
        p = sim_params(grid=(40, 40, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
        reps[r].params, reps[r].ext = p, ext_params(pairPotential=abi.NW_PAIR_WCA, stencil=abi.NW_STENCIL_2D)
        a, b, _ = random_worms(p, rng, twod=True)
        pos.append(a)
        vel.append(b)
    lib.nwBatchSetReplicas(reps, len(sizes))
    P, V = np.concatenate(pos), np.concatenate(vel)
    dP, dV, gP, gV = (DeviceArray.from_numpy(lib, x) for x in (P, V, np.full_like(P, 7), np.full_like(P, 7)))
    out = (ctypes.c_double * len(sizes))()
    lib.nwBatchPolarSpeedGrad(dP.p, dV.p, gP.p, gV.p, out)
    hP, hV, at = gP.download(np.uint32, P.shape), gV.download(np.uint32, P.shape), 0
    for r, (W, n) in enumerate(sizes):
        N = W * n
        lib.setParameters(ctypes.byref(reps[r].params))
        d = [DeviceArray.from_numpy(lib, x) for x in (pos[r], vel[r], np.zeros_like(pos[r]), np.zeros_like(pos[r]))]
        one = lib.nwPolarSpeedGrad(d[0].p, d[1].p, W, d[2].p, d[3].p)
        assert abs(out[r] - one) <= 1e-12 * max(1.0, abs(one))
        assert np.array_equal(hP[at:at + N], d[2].download(np.uint32, (N, 4))), r
        assert np.array_equal(hV[at:at + N], d[3].download(np.uint32, (N, 4))), r
        at += N
    lib.nwBatchSetReplicas(None, 0)
