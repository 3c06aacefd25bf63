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
int network(uint64_t n, uint64_t cells, uint64_t buckets) { return nw::srd_network(n, cells, buckets); }
int late(uint64_t n, uint64_t cells) { return nw::srd_late(n, cells); }
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
    lib.network.argtypes, lib.late.argtypes = [U64, U64, U64], [U64, U64]
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


@pytest.mark.parametrize("per,buckets,network,late", [
    (5, 700, 16, 0), (7, 700, 16, 0), (8, 700, 32, 0), (12, 1024, 32, 0), (13, 1024, 32, 1), (26, 700, 32, 1),
    (27, 700, 16, 1), (80, 700, 16, 1),      # dense cells: by insertion, many workgroups
    (8, 1025, 16, 0), (20, 2048, 16, 1),     # two rounds of the larger network, one of the smaller
    (9, 2049, 16, 0), (10, 2049, 32, 0), (21, 9000, 32, 1), (22, 9000, 16, 1)])
def test_network_of_the_srd_cells(rules, per, buckets, network, late):
    cells = 100_000
    assert (rules.network(per * cells, cells, buckets), rules.late(per * cells, cells)) == (network, late)
