"""The one-launch cell order and pair pass where a workgroup's rows and the rows
beside them outgrow its stage many times over: a band of worms, worms on top
of each other in one cell, rows at the periodic face.  Against the two-level
sort and the pair kernel: bit for bit, and in a time of the same order (the
candidates are the same; passes over the whole system are hundreds of times
more).  A small wcaEpsilon keeps overlapping beads' forces finite."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, NWTuning, timer_read
from nwtest import ext_params, random_forces, random_worms, sim_params
from test_gpu_rows import lib, step  # noqa: F401 (lib: the fixture)

pytestmark = pytest.mark.gpu

MD = ("md_front", "md_tiles", "md_sort", "md_collide")


def crowd(rng, grid, W, n, at, size):
    """Worms in the box's part of `size` (x, y fractions) from `at` on, wrapped."""
    p = sim_params(grid=(*grid, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
    pos, vel, tan = random_worms(p, rng, twod=True)
    for k in range(2):
        L = 1.2 * grid[k]
        x = (pos[:, k].astype(np.float64) + L / 2) * size[k] + at[k] * L
        pos[:, k] = (x % L - L / 2).astype(np.float32)
    f = random_forces(rng, W * n, 0.5)
    f[:, 3] = 0
    return p, (pos, vel, f, f[::-1].copy(), tan)


def ext(**kw):
    return ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0, wcaEpsilon=1e-30,
                      stencil=abi.NW_STENCIL_2D, **kw)


@pytest.mark.parametrize("grid,W,n,at,size,one", [
    ((200, 200), 6400, 10, (0.0, 0.3), (1.0, 0.06), True),    # 12 rows of 5,000 beads
    ((20, 513), 3000, 5, (0.0, 0.98), (1.0, 0.03), True),     # three own rows, across the periodic face
    ((30, 400), 500, 8, (0.2, 0.5), (0.02, 0.002), True),     # 4,000 beads in a cell or two
    ((3, 3), 900, 7, (0.0, 0.0), (1.0, 1.0), False),          # crowded throughout: not taken in one launch
])
def test_crowded_equals_sort_and_pairs(lib, grid, W, n, at, size, one):  # noqa: F811
    p, state = crowd(np.random.default_rng([*grid, W, n]), grid, W, n, at, size)
    ms = []
    got = []
    for t in (NWTuning(), NWTuning(mdMembers=512)):
        step(lib, p, ext(), state, t, 0)  # (LDS grants, scratch)
        for f in MD:
            lib.nwTimerEnable(f.encode(), 1)
        got.append(step(lib, p, ext(), state, t, 0))
        ms.append(sum(timer_read(lib, f)[0] for f in MD))
        if not t.mdMembers:
            assert timer_read(lib, "md_sort")[1] == (0 if one else 2)
        for f in MD:
            lib.nwTimerEnable(f.encode(), 0)
    print(f"{grid} {W * n}: {ms[0] / 2 * 1e3:.0f} us a step, sort and pair kernel {ms[1] / 2 * 1e3:.0f}", flush=True)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "hash", "ids", "sortedPos"), *got):
        assert np.array_equal(x, y), (name, int((x != y).sum()))
    assert ms[0] < 20 * ms[1], ms


def test_crowded_batch(lib):  # noqa: F811
    rng = np.random.default_rng(11)
    parts = [((9, 12), 20, 9, (0, 0), (1, 1)), ((200, 200), 3200, 10, (0, 0.97), (1, 0.03)),
             ((20, 300), 1500, 5, (0, 0.3), (1, 0.03)), ((12, 9), 200, 6, (0.1, 0.1), (0.1, 0.1))]
    reps, states = (abi.NWReplicaParams * len(parts))(), []
    for r, q in enumerate(parts):
        reps[r].params, state = crowd(rng, *q)
        reps[r].seed = 5 + r
        states.append(state)
    arrays = [np.concatenate([s[k] for s in states]) for k in range(5)]
    N, got = len(arrays[0]), []
    for kern in (abi.NW_COLLIDE_AUTO, abi.NW_COLLIDE_LDS):
        for r in range(len(parts)):
            reps[r].ext = ext(collideKernel=kern)
        lib.nwBatchSetReplicas(reps, len(parts))
        d = [DeviceArray.from_numpy(lib, x) for x in arrays]
        i, sp = DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
        lib.nwTimerEnable(b"batch_sort", 1)
        lib.nwBatchMdStep(*[x.p for x in d], i.p, sp.p, None, None, 1e-4, 2, 0)
        assert timer_read(lib, "batch_sort")[1] == (0 if kern == abi.NW_COLLIDE_AUTO else 2)
        lib.nwTimerEnable(b"batch_sort", 0)
        assert lib.nwGetLastError() == 0
        got.append([x.download(np.uint32, (N, 4)) for x in d] + [i.download(np.uint32, (N,)),
                                                                 sp.download(np.uint32, (N, 4))])
    lib.nwBatchSetReplicas(None, 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "ids", "sortedPos"), *got):
        assert np.array_equal(x, y), name



def test_crowded_without_allocation(lib):  # noqa: F811
    """The same through nwFusedMdStepNoAlloc, whose crowded rows have their place in its fixed scratch."""
    p, state = crowd(np.random.default_rng(5), (200, 200), 3200, 10, (0.0, 0.98), (1.0, 0.04))
    N = p.numParticles
    want = step(lib, p, ext(), state, NWTuning(mdMembers=512), 0)
    lib.nwSetTuning(ctypes.byref(NWTuning()))
    d = [DeviceArray.from_numpy(lib, a) for a in state]
    i, sp = DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
    lib.nwRngSetSeed(11, 5)
    for _ in range(2):
        lib.nwFusedMdStepNoAlloc(*[x.p for x in d], None, i.p, sp.p, None, None, 1e-4, 2.0, 0.1, 1, p.numFilaments)
    assert lib.nwGetLastError() == 0, lib.nwGetLastErrorString()
    got = [x.download(np.uint32, (N, 4)) for x in d] + [i.download(np.uint32, (N,)), sp.download(np.uint32, (N, 4))]
    for x, y in zip(got, want[:5] + want[6:]):
        assert np.array_equal(x, y)
