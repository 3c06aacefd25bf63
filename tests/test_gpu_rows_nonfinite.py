"""Worms with beads at NaN or infinity (a run that blew up, a caller's hole in
the data) in the one-launch cell order and pair pass, alone and in a batch,
against the two-level sort and the pair kernel.  Such a bead hashes to some cell
of the grid, adds nothing to its neighbours' pair forces and passes its value
on along its worm: every output is the same, bit for bit where it is a number
and NaN where the other is NaN (the payload of a NaN is not compared)."""
import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, NWTuning
from nwtest import ext_params, random_forces, random_worms, sim_params
from test_gpu_rows import lib, step  # noqa: F401 (lib: the fixture)

pytestmark = pytest.mark.gpu

NAN, INF = np.float32(np.nan), np.float32(np.inf)
HOLES = [(0, 0, NAN), (1, 1, NAN), (1, 0, INF), (2, 0, -INF), (2, 1, INF), (3, 1, -INF), (4, 2, NAN), (5, 2, INF)]


def system(rng, grid, W, n):
    p = sim_params(grid=(*grid, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
    pos, vel, tan = random_worms(p, rng, twod=True)
    f = random_forces(rng, W * n, 0.5)
    f[:, 3] = 0
    for k, axis, x in HOLES:
        bead = (k * (W // 6) * n + (2 * k) % n) % (W * n)
        pos[bead, axis] = x
        vel[(bead + 3 * n) % (W * n), 0] = x
    return p, (pos, vel, f, f[::-1].copy(), tan)


def ext(**kw):
    return ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                      stencil=abi.NW_STENCIL_2D, **kw)


def same(a, b):
    nan = np.isnan(a.view(np.float32)) & np.isnan(b.view(np.float32)) if a.ndim == 2 else np.zeros(a.shape, bool)
    return bool(np.all((a == b) | nan))


@pytest.mark.parametrize("grid,W,n", [((64, 64), 333, 7), ((31, 300), 400, 13), ((40, 3), 21, 11), ((190, 190), 3000, 12)])
def test_nonfinite_beads(lib, grid, W, n):  # noqa: F811
    p, state = system(np.random.default_rng([*grid, W, n]), grid, W, n)
    a = step(lib, p, ext(), state, NWTuning(), 0)
    b = step(lib, p, ext(), state, NWTuning(mdMembers=512), 0)
    assert np.isnan(a[0].view(np.float32)).any() and np.isfinite(a[2].view(np.float32)).mean() > 0.2
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "hash", "ids", "sortedPos"), a, b):
        assert same(x, y), name
    assert np.array_equal(a[6], np.argsort(a[5], kind="stable"))


def test_nonfinite_beads_in_a_batch(lib):  # noqa: F811
    rng = np.random.default_rng(3)
    parts = [((12, 9), 30, 6), ((64, 64), 333, 7), ((9, 300), 200, 9)]
    reps, states = (abi.NWReplicaParams * len(parts))(), []
    for r, q in enumerate(parts):
        reps[r].params, state = system(rng, *q)
        states.append(state)
    arrays = [np.concatenate([s[k] for s in states]) for k in range(5)]
    N, got = len(arrays[0]), []
    for kern in (abi.NW_COLLIDE_AUTO, abi.NW_COLLIDE_LDS):
        for r in range(len(parts)):
            reps[r].ext = ext(collideKernel=kern)
        lib.nwBatchSetReplicas(reps, len(parts))
        d = [DeviceArray.from_numpy(lib, x) for x in arrays]
        i, sp = DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
        lib.nwBatchMdStep(*[x.p for x in d], i.p, sp.p, None, None, 1e-4, 2, 0)
        assert lib.nwGetLastError() == 0
        got.append([x.download(np.uint32, (N, 4)) for x in d] + [i.download(np.uint32, (N,)),
                                                                 sp.download(np.uint32, (N, 4))])
    lib.nwBatchSetReplicas(None, 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "ids", "sortedPos"), *got):
        assert same(x, y), name
