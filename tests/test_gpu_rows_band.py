"""Bands of worms that outgrow a workgroup's stage in the one-launch cell order
and pair pass, while the two rows beside its own fit it (or only just): the
step against the two-level sort and the pair kernel, bit for bit."""
import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, NWTuning
from nwtest import ext_params, random_forces, random_worms, sim_params
from test_gpu_rows import lib, step  # noqa: F401 (lib: the fixture)

pytestmark = pytest.mark.gpu


def band(rng, grid, W, n, at, height):
    """Worms in the rows' part [at, at + height) of the box, wrapped."""
    p = sim_params(grid=(*grid, 1), cell=1.2, W=W, n=n, bondSpringL=0.8, activity=0.0)
    pos, vel, tan = random_worms(p, rng, twod=True)
    L = 1.2 * grid[1]
    y = (pos[:, 1].astype(np.float64) + L / 2) * height + at * L
    pos[:, 1] = (y % L - L / 2).astype(np.float32)
    f = random_forces(rng, W * n, 0.5)
    f[:, 3] = 0
    return p, (pos, vel, f, f[::-1].copy(), tan)


@pytest.mark.parametrize("grid,W,n,at,height", [
    ((20, 513), 1400, 5, 0.3, 0.045),  # three own rows, about 300 beads a row against a stage of 1,024
    ((20, 513), 1400, 5, 0.98, 0.045),  # across the periodic face
    ((64, 64), 800, 10, 0.4, 0.25),    # one own row, the rows beside it at the stage's edge
])
def test_band_equals_sort_and_pairs(lib, grid, W, n, at, height):  # noqa: F811
    rng = np.random.default_rng([*grid, W, n])
    p, state = band(rng, grid, W, n, at, height)
    e = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                   stencil=abi.NW_STENCIL_2D)
    a = step(lib, p, e, state, NWTuning(), 0)
    b = step(lib, p, e, state, NWTuning(mdMembers=512), 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "hash", "ids", "sortedPos"), a, b):
        assert np.array_equal(x, y), (name, int((x != y).sum()))


def test_band_in_a_batch(lib):  # noqa: F811
    rng = np.random.default_rng(7)
    parts = [((9, 12), 20, 9, 0.1, 1.0), ((20, 513), 1400, 5, 0.98, 0.045), ((9, 300), 700, 9, 0.3, 0.06)]
    reps, states = (abi.NWReplicaParams * len(parts))(), []
    for r, q in enumerate(parts):
        reps[r].params, state = band(rng, *q)
        reps[r].seed = 5 + r
        states.append(state)
    arrays = [np.concatenate([s[k] for s in states]) for k in range(5)]
    N, got = len(arrays[0]), []
    for kern in (abi.NW_COLLIDE_AUTO, abi.NW_COLLIDE_LDS):
        for r in range(len(parts)):
            reps[r].ext = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                                     stencil=abi.NW_STENCIL_2D, collideKernel=kern)
        lib.nwBatchSetReplicas(reps, len(parts))
        d = [DeviceArray.from_numpy(lib, x) for x in arrays]
        i, sp = DeviceArray(lib, 4 * N), DeviceArray(lib, 16 * N)
        lib.nwBatchMdStep(*[x.p for x in d], i.p, sp.p, None, None, 1e-4, 2, 0)
        lib.threadSync()
        assert lib.nwGetLastError() == 0
        got.append([x.download(np.uint32, (N, 4)) for x in d] + [i.download(np.uint32, (N,)),
                                                                 sp.download(np.uint32, (N, 4))])
    lib.nwBatchSetReplicas(None, 0)
    for name, x, y in zip(("pos", "vel", "force", "forceOld", "tangent", "ids", "sortedPos"), *got):
        assert np.array_equal(x, y), name
