"""A refused nwBatchSetReplicas leaves the batch before it whole: its layout, its
generator offsets, its steps (bit for bit those of a batch set once) and its
adjoint, whether a replica's worms or its grid are refused."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, lattice_system_2d, sim_params

pytestmark = pytest.mark.gpu

R = 3


def replicas():
    reps, pos, vel = (abi.NWReplicaParams * R)(), [], []
    for r in range(R):
        p, a, b = lattice_system_2d(40 + 7 * r, 9, 34, np.random.default_rng(r))
        p.gamma = 2.0
        reps[r].params, reps[r].seed, reps[r].offset, reps[r].langevin = p, 9 + r, 100 + r, 1
        reps[r].langevinGamma, reps[r].langevinKbT = 2.0, 5.0
        reps[r].ext = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=3.0,
                                 stencil=abi.NW_STENCIL_2D)
        pos.append(a)
        vel.append(b)
    return reps, np.concatenate(pos), np.concatenate(vel)


def refused(lib, what):
    reps = (abi.NWReplicaParams * 1)()
    reps[0].params = sim_params(grid=(34, 34, 1), cell=1.2, W=4, n=65) if what == "worms" else sim_params(
        grid=(9000, 9000, 1), cell=1.2, W=4, n=9, activity=0.0)  # 81 million cells: more buckets than the sort takes
    reps[0].ext = ext_params(pairPotential=abi.NW_PAIR_WCA, stencil=abi.NW_STENCIL_2D)
    lib.nwBatchSetReplicas(reps, 1)
    assert lib.nwGetLastError() == -22


@pytest.mark.parametrize("what", ["worms", "grid"])
def test_refused_batch_leaves_the_one_before(nwlib, what):
    lib = nwlib
    reps, pos, vel = replicas()
    N, got = len(pos), []
    try:
        for refuse in (False, True):
            lib.nwBatchSetReplicas(reps, R)
            if refuse:
                refused(lib, what)
            off = (ctypes.c_uint64 * 1)()
            for r in range(R):
                lib.nwBatchRngState(r, off)
                assert off[0] == 100 + r
            b, c = np.zeros(R + 1, np.uint32), np.zeros(R + 1, np.uint32)
            lib.nwBatchLayout(b.ctypes.data, c.ctypes.data)
            assert b[-1] == N and c[-1] == R * 34 * 34
            d = [DeviceArray.from_numpy(lib, x) for x in (pos, vel, *[np.zeros_like(pos)] * 3)]
            w = [DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)]
            lib.nwBatchMdStep(*[x.p for x in d], w[0].p, w[1].p, None, None, 1e-3, 3, 0)
            if refuse:
                refused(lib, what)
            lib.nwBatchAdjointForward(*[x.p for x in d], 1e-3, 0, None, 3, 2)
            if refuse:
                refused(lib, what)
            g = (ctypes.c_double * (4 * R))()
            ones = DeviceArray.from_numpy(lib, np.ones_like(pos))
            lib.nwBatchAdjointBackward(ones.p, None, g)
            assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
            got.append([x.download(np.uint32, (N, 4)) for x in d] + [np.array(g)])
    finally:
        lib.nwBatchSetReplicas(None, 0)
    for x, y in zip(*got):
        assert np.array_equal(x, y)
