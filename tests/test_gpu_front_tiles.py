"""The front that also does the sort's first level against the two launches
(asked for by a front workgroup of 256): worms of one bead to a whole
wavefront, a single worm, whole and ragged last tiles of both workgroup sizes
and the last size that takes it.  Every output bit for bit."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray
from nwtest import ext_params, random_forces, random_worms, sim_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,n,dem", [
    (1, 1, 1), (1, 64, 1), (513, 1, 1), (8 * 4, 13, 1), (8 * 4 + 1, 13, 0), (8 * 9 - 1, 33, 0),
    (2048 * 2, 31, 0), (2048 * 2 + 1, 31, 1), (2049, 64, 0), (4096 * 3, 20, 0), (4096 * 3 + 1, 20, 0), (700, 10, 1)])
def test_one_launch_equals_two(nwlib, W, n, dem):
    lib, rng, N = nwlib, np.random.default_rng([W, n]), W * n
    G = max(6, int(np.ceil((N / 0.5) ** 0.5)))
    p = sim_params(grid=(max(4, int(N ** (1 / 3))),) * 3 if dem else (G, G, 1), cell=1.2, W=W, n=n, bondSpringL=0.8,
                   activity=0.4)
    p.reverseProbability, p.gamma = 0.2, 2.0
    e = ext_params(driveForce=1.0) if dem else ext_params(pairPotential=abi.NW_PAIR_WCA, driveForce=1.0,
                                                          bondedMode=abi.NW_BONDED_CHAIN, stencil=abi.NW_STENCIL_2D)
    pos, vel, tan = random_worms(p, rng, twod=not dem)
    f = random_forces(rng, N, 0.5)
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    out = []
    try:
        for block in (0, 256):
            t = abi.NWTuning()
            t.frontBlock = block
            lib.nwSetTuning(ctypes.byref(t))
            lib.nwRngSetSeed(3, 40)
            d = [DeviceArray.from_numpy(lib, x) for x in (pos, vel, f, f, tan)]
            u = [DeviceArray(lib, 4 * N) for _ in range(2)]
            s = [DeviceArray(lib, 16 * N) for _ in range(3)]
            lib.nwFusedMdStep(*[x.p for x in d], u[0].p, u[1].p, s[0].p, s[1].p if dem else None, s[2].p, 1e-3, 2.0,
                              50.0, 1, W)
            out.append([x.download(np.uint32, (N, 4)) for x in (*d, s[0], s[2])] + [x.download(np.uint32, (N,)) for x in u])
    finally:
        lib.nwSetTuning(ctypes.byref(abi.NWTuning()))
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), k
    assert np.array_equal(out[0][-1], np.argsort(out[0][-2], kind="stable"))
