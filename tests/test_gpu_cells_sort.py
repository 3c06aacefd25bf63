"""The cell sort's second level at its edges: one member, a bucket filled to
and past each stage (1,024 and 2,048 members), one cell holding a whole
bucket, a last bucket whose cell count is no multiple of four, more tiles
than threads.  Equal to a stable sort by key, exactly."""
import numpy as np
import pytest

from nwamd.abi import DeviceArray

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
