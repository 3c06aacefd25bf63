"""The cell sort's second level at its edges: one member, a bucket filled to
and past each stage (1,024 and 2,048 members), one cell holding a whole
bucket, a last bucket whose cell count is no multiple of four, more tiles
than threads.  Equal to a stable sort by key, exactly."""
import ctypes

import numpy as np
import pytest

from nwamd.abi import DeviceArray
from nwtest import ext_params, sim_params, solvent_params

pytestmark = pytest.mark.gpu


def spread(n, bound, rng):
    return rng.integers(0, bound, n)


def one_cell(n, bound, rng):
    return np.full(n, bound - 1)


def one_bucket(members):
    # the first `members` keys (shuffled in) below 64, the rest from 4,096 up
    def keys(n, bound, rng):
        k = rng.integers(4096, bound, n)
        k[rng.permutation(n)[:members]] = rng.integers(0, 64, members)
        return k
    return keys


@pytest.mark.parametrize("n,bound,keys", [
    (1, 1, one_cell), (2, 3, spread), (2048, 1, one_cell), (2049, 1, one_cell),
    (2000, 8192, one_cell), (2000, 8192, one_bucket(1024)), (2000, 8192, one_bucket(1025)),
    (5000, 2047, spread), (5000, 1537, spread), (30_000, 29_999, spread), (300_001, 250_003, spread),
    (2_200_000, 2_000_003, spread)])
def test_equals_stable_sort(nwlib, n, bound, keys):
    rng = np.random.default_rng([n, bound])
    k = keys(n, bound, rng).astype(np.uint32)
    v = rng.permutation(n).astype(np.uint32)
    dk, dv = DeviceArray.from_numpy(nwlib, k), DeviceArray.from_numpy(nwlib, v)
    nwlib.nwSortParticlesBounded(dk.p, dv.p, n, bound)
    o = np.argsort(k, kind="stable")
    assert np.array_equal(dk.download(np.uint32, (n,)), k[o])
    assert np.array_equal(dv.download(np.uint32, (n,)), v[o])


@pytest.mark.parametrize("Ns,heap", [(1, 0), (7 * 1024, 0), (7 * 1024 + 1, 0), (20_000, 40), (3000, 20), (3_000_000, 40)])
def test_srd_cells(nwlib, Ns, heap):
    """The collision's cells on either side of seven particles a cell, with cells of `heap` particles more (past either
    sorting network), and with more tiles than threads: the order of a stable sort by cell exactly, the cells' mean
    velocities against sums in FP64 (a mean of at most a few hundred FP32 terms: 1e-5 of the speeds)."""
    lib, rng = nwlib, np.random.default_rng([Ns, heap])
    L = 32 if Ns < 1_000_000 else 512
    p = sim_params(grid=(L, L, 1), cell=1.0, W=1, n=3)
    s = solvent_params(p, (L, L, 1), (1.0, 1.0, 1.0), alpha=1.0, kbT=0.3, offset=(0.0, 0.0, 0.0), ns=Ns)
    NT = 3 + Ns
    pos, vel = np.zeros((NT, 4), np.float32), np.zeros((NT, 4), np.float32)
    pos[:, :2] = (rng.random((NT, 2)) - 0.5) * L * 0.999
    if heap:
        for c in (3.5, -7.5):
            pos[rng.choice(NT, heap, replace=False), :2] = c
    pos[:, 2] = p.origin.z + 0.5
    vel[:, :2] = rng.normal(0, 1, (NT, 2))
    vel[:, 3] = 1.0
    lib.setParameters(ctypes.byref(p))
    lib.setSolventParameters(ctypes.byref(s))
    lib.nwSetExtParameters(ctypes.byref(ext_params(srdCollideFilaments=1)))
    P, V = DeviceArray.from_numpy(lib, pos), DeviceArray.from_numpy(lib, vel)
    h, i, com = DeviceArray(lib, 4 * NT), DeviceArray(lib, 4 * NT), DeviceArray(lib, 16 * L * L)
    lib.nwFusedSrdStep(P.p, V.p, com.p, h.p, i.p, 0.01, 3, Ns, 0)
    hash_, ids = h.download(np.uint32, (NT,)), i.download(np.uint32, (NT,))
    assert np.array_equal(ids, np.argsort(hash_, kind="stable"))
    n = np.bincount(hash_, minlength=L * L)
    mean = np.stack([np.bincount(hash_, vel[:, k].astype(np.float64), L * L) for k in range(3)], 1) / np.maximum(n, 1)[:, None]
    assert np.abs(com.download(np.float32, (L * L, 4))[:, :3] - mean).max() < 5e-5
