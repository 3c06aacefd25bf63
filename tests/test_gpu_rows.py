"""The one-launch cell order and pair pass of small systems (nw_rows.hip),
the built-in choice, against the two-level sort and the pair kernel that an
explicit launch shape asks for: positions, velocities, forces, cell order,
cells and sorted records bit for bit, at the edges of its grids, with cells at
an address that is not a multiple of 16, and with rows so full that a
workgroup's beads do not fit its LDS."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, NWTuning
from nwtest import ext_params, random_forces, random_worms, sim_params

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib(nwlib):
    yield nwlib
    nwlib.nwSetTuning(ctypes.byref(NWTuning()))


def step(lib, p, e, state, tuning, shift):
    lib.nwSetTuning(ctypes.byref(tuning))
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    N = p.numParticles
    d = [DeviceArray.from_numpy(lib, a) for a in state]
    h, i, sp = DeviceArray(lib, 4 * (N + 4)), DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
    lib.nwRngSetSeed(11, 5)
    for _ in range(2):
        lib.nwFusedMdStep(*[x.p for x in d], ctypes.c_void_p(h.p.value + 4 * shift), i.p, sp.p, None, None, 1e-4, 2.0,
                          0.1, 1, p.numFilaments)
    lib.threadSync()
    assert lib.nwGetLastError() == 0
    return [x.download(np.uint32, (N, 4)) for x in d] + [h.download(np.uint32, (N,), 4 * shift),
                                                         i.download(np.uint32, (N,)), sp.download(np.uint32, (N, 4))]


@pytest.mark.parametrize("grid,W,n,shift,squeeze", [
    ((3, 3), 1, 1, 0, 1.0),         # one bead, every stencil the whole grid
    ((3, 3), 5, 7, 1, 1.0),         # every cell an edge, words before the first whole group of four
    ((5, 4), 3, 9, 2, 1.0),
    ((40, 3), 21, 11, 3, 1.0),      # three rows: a workgroup stages the whole grid
    ((64, 64), 333, 7, 0, 1.0),
    ((64, 64), 333, 7, 3, 1.0),
    ((31, 300), 400, 13, 0, 1.0),   # two rows a workgroup
    ((20, 513), 700, 5, 1, 1.0),    # three rows a workgroup, the last one ragged
    ((64, 64), 800, 10, 0, 0.04),   # every bead in three rows: past the stage
    ((200, 200), 3700, 10, 1, 0.015),  # and past the list of groups
])
def test_one_launch_equals_sort_and_pairs(lib, grid, W, n, shift, squeeze):
    rng = np.random.default_rng([*grid, W, n, shift])
    p = sim_params(grid=(*grid, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
    e = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                   stencil=abi.NW_STENCIL_2D)
    pos, vel, tan = random_worms(p, rng, twod=True)
    pos[:, 1] = (pos[:, 1].astype(np.float64) * squeeze).astype(np.float32)
    f = random_forces(rng, W * n, 0.5)
    f[:, 3] = 0
    state = (pos, vel, f, f[::-1].copy(), tan)
    a = step(lib, p, e, state, NWTuning(), shift)
    b = step(lib, p, e, state, NWTuning(mdMembers=512), shift)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "hash", "ids", "sortedPos"), a, b):
        assert np.array_equal(x, y), (name, int((x != y).sum()))


@pytest.mark.parametrize("sizes", [
    [(1, 1, 3), (5, 7, 3), (40, 16, 31), (3, 5, 4), (333, 7, 64), (17, 12, 300)],  # uneven, offsets of every residue
    [(20, 9, 12)] * 40,                                                            # more rows than workgroups wanted
])
def test_batch_one_launch_equals_sort_and_pairs(lib, sizes):
    """Replicas (worms, beads per worm, cells a side) stepped together: the built-in choice against the sort and the
    pair kernel (collideKernel set), forces, positions, cell order and sorted records bit for bit."""
    rng = np.random.default_rng([29, len(sizes)])
    reps, pos, vel, force = (abi.NWReplicaParams * len(sizes))(), [], [], []
    for r, (W, n, G) in enumerate(sizes):
        p = sim_params(grid=(G, G, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
        q = random_worms(p, rng, twod=True)
        f = random_forces(rng, W * n, 0.5)
        f[:, 3] = 0
        reps[r].params, reps[r].seed, reps[r].offset, reps[r].langevin = p, 7 + r, 3, 1
        reps[r].langevinGamma, reps[r].langevinKbT = p.gamma, 0.1
        pos.append(q[0])
        vel.append(q[1])
        force.append(f)
    arrays = [np.concatenate(x) for x in (pos, vel, force, force[::-1], force)]
    N = len(arrays[0])
    got = []
    for kern in (abi.NW_COLLIDE_AUTO, abi.NW_COLLIDE_LDS):
        for r in range(len(sizes)):
            reps[r].ext = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                                     stencil=abi.NW_STENCIL_2D, collideKernel=kern)
        lib.nwBatchSetReplicas(reps, len(sizes))
        d = [DeviceArray.from_numpy(lib, a) for a in arrays]
        i, sp = DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
        for graph in (0, 1):
            lib.nwBatchMdStep(*[x.p for x in d], i.p, sp.p, None, None, 1e-4, 3, graph)
        lib.threadSync()
        assert lib.nwGetLastError() == 0
        got.append([x.download(np.uint32, (N, 4)) for x in d] + [i.download(np.uint32, (N,)),
                                                                 sp.download(np.uint32, (N, 4))])
    lib.nwBatchSetReplicas(None, 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "ids", "sortedPos"), *got):
        assert np.array_equal(x, y), name
