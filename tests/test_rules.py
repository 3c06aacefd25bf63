"""The rules of the launches' dispatch (nw_rules.hpp), compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D, U32, U64 = ctypes.c_double, ctypes.c_uint32, ctypes.c_uint64
C = """#include "nw_rules.hpp"
extern "C" {
double packed(double area, double sigma, double bond) { return nw::worms_packed(area, sigma, bond); }
int lanes(uint64_t beads, int oneLayer) { return nw::pair_lanes(beads, oneLayer != 0); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text(C)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", f"{ROOT}/nematic-worms_amd/csrc",
                    str(d / "r.cpp"), "-o", str(d / "r.so")], check=True)
    lib = ctypes.CDLL(str(d / "r.so"))
    lib.packed.restype, lib.packed.argtypes = D, [D, D, D]
    lib.lanes.argtypes = [U64, ctypes.c_int]
    return lib


def nearest(d, h):
    """Least distance between beads of neighbouring rows of spacing d at distance h, the rows half a spacing apart."""
    return np.hypot(d / 2, h)


@pytest.mark.parametrize("sigma", [0.5, 1.0, 2.0])
@pytest.mark.parametrize("bond", [0.3, 0.8, 1.0, 1.7])
def test_packing_of_worms(rules, sigma, bond):
    """The densest rows in which beads of different worms keep sigma: found by bisection of the rows' distance."""
    d = min(max(bond, 0.25 * sigma), sigma)
    lo, hi = 0.0, 2 * sigma
    for _ in range(60):
        h = (lo + hi) / 2
        lo, hi = (lo, h) if nearest(d, h) >= sigma else (h, hi)
    area = 1.44 * sigma * sigma
    assert rules.packed(area, sigma, bond) == pytest.approx(min(area / (d * hi), 16.0), rel=1e-9)


def test_packing_limits(rules):
    assert rules.packed(1.2599, 1.0, 1.0) == pytest.approx(1.455, rel=1e-3)  # hexagonal, a cell of the WCA range
    assert rules.packed(1.44, 1.0, 0.8) > 1.75  # bonds of 0.8 sigma: a band of 1.75 a cell stays in the stage
    assert rules.packed(1.44, 0.0, 0.8) == 16.0 and rules.packed(1.44, 1.0, 0.0) <= 16.0


@pytest.mark.parametrize("beads,layer,layers", [(1, 8, 8), (200_000, 8, 8), (200_001, 2, 4), (1 << 31, 2, 4)])
def test_lanes_of_the_pair_list(rules, beads, layer, layers):
    assert (rules.lanes(beads, 1), rules.lanes(beads, 0)) == (layer, layers)
