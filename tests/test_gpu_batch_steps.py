"""A batch call of several steps against as many calls of one step: the call's
last step leaves forces, old forces and tangents where the caller reads them,
for odd and even step counts, direct and replayed, with and without reversal
(which moves the old forces) and the extensile term (which reads tangents).
Bit for bit."""
import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, lattice_system_2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reverse,activity,n", [(0.0, 0.0, 9), (0.0, 0.0, 3), (0.3, 0.0, 9), (0.0, 2.0, 9)])
@pytest.mark.parametrize("graph", [0, 1])
def test_steps_in_one_call(nwlib, reverse, activity, n, graph):
    lib, R = nwlib, 3
    reps, pos, vel = (abi.NWReplicaParams * R)(), [], []
    for r in range(R):
        p, a, b = lattice_system_2d(40 + 7 * r, n, 34, np.random.default_rng([n, r]))
        p.gamma, p.reverseProbability, p.activity = 2.0, reverse, activity
        reps[r].params, reps[r].seed, reps[r].offset, reps[r].langevin = p, 9 + r, 5, 1
        reps[r].ext = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=3.0,
                                 stencil=abi.NW_STENCIL_2D)
        reps[r].langevinGamma, reps[r].langevinKbT = 2.0, 50.0
        pos.append(a)
        vel.append(b)
    start = [np.concatenate(x) for x in (pos, vel)]
    N = start[0].shape[0]

    def run(calls, graph):
        lib.nwBatchSetReplicas(reps, R)
        d = [DeviceArray.from_numpy(lib, x) for x in (*start, *[np.zeros_like(start[0])] * 3)]
        w = [DeviceArray.from_numpy(lib, np.zeros((N, 4), np.float32)) for _ in range(4)]
        for steps in calls:
            lib.nwBatchMdStep(*[x.p for x in d], w[0].p, w[1].p, w[2].p, w[3].p, 1e-3, steps, graph)
        return [x.download(np.float32, (N, 4)) for x in d]

    for calls in ([1], [2], [3], [4], [3, 3], [2, 4, 1], [5, 2]):
        one = run([1] * sum(calls), 0)
        for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent"), run(calls, graph), one):
            assert np.array_equal(x, y), (calls, name)
    lib.nwBatchSetReplicas(None, 0)
