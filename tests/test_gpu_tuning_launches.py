"""The autotuner against the launches of small systems: the built-in choice
does cell order and pairs, or the front and the sort's first level, in one
launch, which a knob asked for takes apart.  The tuner must see all that a
candidate costs (its pick keeps the launches that are some 40 % faster), and a
stored choice holds for its own physics and kernels alone."""
import ctypes

import numpy as np
import pytest

from nwamd import abi
from nwamd.abi import DeviceArray, NWTuning, timer_read
from nwtest import ext_params, lattice_system_2d, random_worms, sim_params

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib(nwlib):
    yield nwlib
    nwlib.nwSetTuning(ctypes.byref(NWTuning()))


def system(lib, dem=False, activity=0.0):
    rng = np.random.default_rng(5)
    if dem:
        p = sim_params(grid=(24, 24, 24), cell=1.2, W=1000, n=10, bondSpringL=0.8, activity=0.0)
        pos, vel, _ = random_worms(p, rng)
        e = ext_params()
    else:
        p, pos, vel = lattice_system_2d(2000, 16, 220, rng)
        p.activity = activity
        e = ext_params(pairPotential=abi.NW_PAIR_WCA, bondedMode=abi.NW_BONDED_CHAIN, driveForce=1.0,
                       stencil=abi.NW_STENCIL_2D)
    lib.setParameters(ctypes.byref(p))
    lib.nwSetExtParameters(ctypes.byref(e))
    d = [DeviceArray.from_numpy(lib, x) for x in (pos, vel, *[np.zeros_like(pos)] * 3)]
    return p, d


def tune(lib, p, d, cache=b""):
    out = NWTuning()
    rc = lib.nwAutotuneFused(*[x.p for x in d], p.numFilaments, 0, 1e-4, 2.0, 0.0, 0, 1e-2, 0, 5, cache, 1,
                             ctypes.byref(out))
    assert lib.nwGetLastError() == 0
    return rc, out.as_dict()


def launches(lib, p, d, families):
    N = p.numParticles
    u, s = [DeviceArray(lib, 4 * N) for _ in range(2)], [DeviceArray(lib, 16 * N) for _ in range(3)]
    for f in families:
        lib.nwTimerEnable(f.encode(), 1)
    lib.nwFusedMdStep(*[x.p for x in d], *[x.p for x in u], *[x.p for x in s], 1e-4, 2.0, 0.0, 0, p.numFilaments)
    got = [timer_read(lib, f)[1] for f in families]
    for f in families:
        lib.nwTimerEnable(f.encode(), 0)
    return got


@pytest.mark.parametrize("dem,families,expected", [
    (False, ("md_front", "md_tiles", "md_sort", "md_collide"), [1, 0, 0, 1]),
    (True, ("md_front", "md_tiles", "md_sort", "md_collide"), [1, 0, 1, 1])])
def test_pick_keeps_the_faster_launches(lib, dem, families, expected):
    p, d = system(lib, dem)
    assert launches(lib, p, d, families) == expected
    rc, pick = tune(lib, p, d)
    assert rc == 1
    assert launches(lib, p, d, families) == expected, pick


def test_stored_choice_is_of_its_physics_and_kernels(lib, tmp_path):
    cache = tmp_path / "t.txt"
    p, d = system(lib)
    assert tune(lib, p, d, str(cache).encode())[0] == 1
    device, size, values = cache.read_text().splitlines()[0].split("\t")
    assert tune(lib, p, d, str(cache).encode())[0] == 2
    # the same sizes with the extensile term
    p, d = system(lib, activity=2.0)
    assert tune(lib, p, d, str(cache).encode())[0] == 1
    # a line as stored before the kernels were numbered
    old = tmp_path / "old.txt"
    old.write_text("\t".join((device.split("/k")[0], size, "4096 512 0 0 256 256 0")) + "\n")
    p, d = system(lib)
    assert tune(lib, p, d, str(old).encode())[0] == 1
