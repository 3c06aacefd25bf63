"""The adjoint step's two forms (four lanes a bead for small systems, one for
large ones) against each other: a batch with more wavefronts than the first
takes, against each of its replicas alone.  The same FP32 terms in the same
order, so the gradients agree to FP64 summation (1e-9)."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, lattice_system_2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,n,G,copies", [(1500, 20, 190, 3), (700, 33, 180, 2), (2500, 13, 200, 2)])
def test_one_lane_equals_four(nwlib, W, n, G, copies):
    lib = nwlib
    waves = copies * -(-W // (64 // n))
    assert -(-W // (64 // n)) <= 1024 < waves
    reps, pos, vel, lp = (abi.NWReplicaParams * copies)(), [], [], []
    for r in range(copies):
        rng = np.random.default_rng([W, n, r])
        p, a, b = lattice_system_2d(W, n, G, rng)
        p.gamma = 2.0
        e = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0 + r,
                       stencil=abi.NW_STENCIL_2D)
        reps[r].params, reps[r].ext, reps[r].seed, reps[r].offset, reps[r].langevin = p, e, 5 + r, 11, 1
        reps[r].langevinGamma, reps[r].langevinKbT = 2.0, 100.0
        w = rng.normal(0, 1, a.shape).astype(np.float32)
        w[:, 3] = 0
        pos.append(a)
        vel.append(b)
        lp.append(w)
    steps, K, dt = 6, 3, 1e-3
    lib.nwBatchSetReplicas(reps, copies)
    cat = [np.concatenate(x) for x in (pos, vel)]
    d = [DeviceArray.from_numpy(lib, x) for x in (*cat, *[np.zeros_like(cat[0])] * 3)]
    lib.nwBatchAdjointForward(*[x.p for x in d], dt, 0, None, steps, K)
    g = (ctypes.c_double * (4 * copies))()
    dl = DeviceArray.from_numpy(lib, np.concatenate(lp))
    lib.nwBatchAdjointBackward(dl.p, None, g)
    got = np.array(g).reshape(copies, 4)
    for r in range(copies):
        lib.setParameters(ctypes.byref(reps[r].params))
        lib.nwSetExtParameters(ctypes.byref(reps[r].ext))
        lib.nwRngSetSeed(5 + r, 11)
        one = [DeviceArray.from_numpy(lib, x) for x in (pos[r], vel[r], *[np.zeros_like(pos[r])] * 3)]
        lib.nwAdjointForward(*[x.p for x in one], W, dt, 2.0, 100.0, 1, steps, K)
        h = (ctypes.c_double * 4)()
        dl1 = DeviceArray.from_numpy(lib, lp[r])
        lib.nwAdjointBackward(dl1.p, None, h)
        assert np.allclose(got[r], np.array(h), rtol=1e-9, atol=0), (r, got[r], list(h))
    lib.nwBatchSetReplicas(None, 0)
