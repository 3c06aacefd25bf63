"""Which launches the built-in choice takes, by the timers' launch counts: the
one-launch cell order and pairs (no sort), the front with the sort's first
level (no md_tiles), and the separate launches past their limits.  Without
these counts a comparison of a path with the general one could compare the
general one with itself."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, timer_read
from nwtest import ext_params, random_worms, sim_params

pytestmark = pytest.mark.gpu

MD = ("md_front", "md_tiles", "md_sort", "md_collide")
BATCH = ("batch_front", "batch_tiles", "batch_sort", "batch_collide", "batch_step")
ROWS, FRONT_TILES, SEPARATE = [1, 0, 0, 1], [1, 0, 1, 1], [1, 1, 1, 1]


def wca(**kw):
    return ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                      stencil=abi.NW_STENCIL_2D, **kw)


def counted(lib, families, run):
    for f in families:
        lib.nwTimerEnable(f.encode(), 1)
    run()
    n = [timer_read(lib, f)[1] for f in families]
    for f in families:
        lib.nwTimerEnable(f.encode(), 0)
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    return n


def worms(p, rng):
    """Straight worms at random places (their forces do not matter here)."""
    W, n = p.numFilaments, p.filamentSize
    L = np.array([p.boxSize.x, p.boxSize.y, p.boxSize.z])
    x = rng.random((W, 1, 3)) * L + 0.8 * np.arange(n)[None, :, None] * np.array([1.0, 0.0, 0.0])
    pos = np.zeros((W * n, 4), np.float32)
    pos[:, :3] = x.reshape(-1, 3) % L - L / 2
    return pos


@pytest.mark.parametrize("grid,W,n,e,activity,expected", [
    # the shapes that test_gpu_rows, _band and _worms compare with the sort and the pair kernel
    ((3, 3, 1), 1, 1, wca(), 0.0, ROWS), ((3, 3, 1), 5, 7, wca(), 0.0, ROWS), ((5, 4, 1), 3, 9, wca(), 0.0, ROWS),
    ((40, 3, 1), 21, 11, wca(), 0.0, ROWS), ((64, 64, 1), 333, 7, wca(), 0.0, ROWS),
    ((31, 300, 1), 400, 13, wca(), 0.0, ROWS), ((20, 513, 1), 700, 5, wca(), 0.0, ROWS),
    ((200, 200, 1), 3700, 10, wca(), 0.0, ROWS), ((20, 513, 1), 1400, 5, wca(), 0.0, ROWS),
    # its limits: beads, worms, the term, a launch shape's kernel asked for
    ((600, 600, 1), 16_384, 16, wca(), 0.0, ROWS), ((600, 600, 1), 16_385, 16, wca(), 0.0, ROWS),
    ((700, 700, 1), 13_043, 23, wca(), 0.0, ROWS), ((700, 700, 1), 13_044, 23, wca(), 0.0, SEPARATE),
    ((600, 600, 1), 13_043, 23, wca(), 0.0, SEPARATE),  # 1,500 beads a workgroup
    ((300, 300, 1), 24_576, 3, wca(), 0.0, ROWS), ((300, 300, 1), 24_577, 3, wca(), 0.0, FRONT_TILES),
    ((64, 64, 1), 333, 7, wca(), 0.3, FRONT_TILES), ((2, 64, 1), 33, 7, wca(), 0.0, FRONT_TILES),
    ((64, 64, 1), 333, 7, wca(collideKernel=abi.NW_COLLIDE_LDS), 0.0, FRONT_TILES),
    # the front with the first level: 4,096 wavefronts
    ((24, 24, 24), 700, 10, ext_params(), 0.0, FRONT_TILES), ((64, 64, 64), 4096 * 3, 20, ext_params(), 0.0, FRONT_TILES),
    ((64, 64, 64), 4096 * 3 + 1, 20, ext_params(), 0.0, SEPARATE)])
def test_single_system(nwlib, grid, W, n, e, activity, expected):
    lib, N = nwlib, W * n
    p = sim_params(grid=grid, cell=1.2, W=W, n=n, bondSpringL=0.8, activity=activity)
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    pos = worms(p, np.random.default_rng([W, n]))
    d = [DeviceArray.from_numpy(lib, x) for x in (pos, *[np.zeros_like(pos)] * 4)]
    u, s = [DeviceArray(lib, 4 * N) for _ in range(2)], [DeviceArray(lib, 16 * N) for _ in range(3)]
    assert counted(lib, MD, lambda: lib.nwFusedMdStep(*[x.p for x in (*d, *u, *s)], 0.0, 2.0, 0.0, 0, W)) == expected


@pytest.mark.parametrize("sizes,e,one", [
    ([(1, 1, 3), (5, 7, 3), (40, 16, 31), (3, 5, 4), (333, 7, 64), (17, 12, 300)], wca(), True),
    ([(20, 9, 12)] * 40, wca(), True),
    ([(20, 9, 12)] * 40, wca(collideKernel=abi.NW_COLLIDE_LDS), False),
    ([(2500, 20, 260)] * 14, wca(), True), ([(2501, 20, 260)] * 14, wca(), False),  # 700,000 beads
    ([(5000, 20, 400)] * 2, wca(), True), ([(5001, 20, 400)] * 2, wca(), False)])   # 100,000 a replica
@pytest.mark.parametrize("graph", [0, 1])
def test_batch(nwlib, sizes, e, one, graph):
    lib, R, steps = nwlib, len(sizes), 3
    reps, pos = (abi.NWReplicaParams * R)(), []
    for r, (W, n, G) in enumerate(sizes):
        reps[r].params = sim_params(grid=(G, G, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
        reps[r].ext = e
        pos.append(worms(reps[r].params, np.random.default_rng([W, n, r])))
    pos = np.concatenate(pos)
    d = [DeviceArray.from_numpy(lib, x) for x in (pos, *[np.zeros_like(pos)] * 4)]
    i, sp = DeviceArray(lib, 4 * len(pos)), DeviceArray(lib, 16 * len(pos))
    lib.nwBatchSetReplicas(reps, R)
    got = counted(lib, BATCH, lambda: lib.nwBatchMdStep(*[x.p for x in d], i.p, sp.p, None, None, 0.0, steps, graph))
    lib.nwBatchSetReplicas(None, 0)
    assert got == ([steps, 0, 0, steps, steps] if one else [steps] * 5)
