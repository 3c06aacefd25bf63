// nw_rules.hpp -- rules of the launches' dispatch, as plain host functions of
// sizes and parameters (no HIP in here: the CPU tests compile this file).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace nw {

// Beads of repelling worms that one square of `area` holds at most: rows of
// beads at the bond's length side by side, each bead in the gap between two of
// the next row (the hexagonal packing where the bond is no shorter than
// sigma; beads of a worm do not repel each other).
inline double worms_packed(double area, double sigma, double bond) {
    const double d = std::max(std::min(bond, sigma), 0.25 * sigma);
    if (!(d > 0.0)) return 16.0;  // nothing keeps them apart
    return std::min(area / (d * std::sqrt(sigma * sigma - 0.25 * d * d)), 16.0);
}

// Lanes that share a bead in the pair list (nw_pairs.hip): 8 while that fills
// the chip; beyond, the lanes' lookups and sums are work: 2 where the stencil
// is 9 cells, 4 where it is 27.  Through the tables, us, beads in rows (evenly
// filled cells, the state that a run settles in) / worms at random places
// (cells of many beads beside empty ones, where one lane waits for its
// fullest), one lane a bead without a list / 8 (the soft spheres) or 4 lanes
// with 64 entries a list / 2 lanes with 24:
//   one layer, WCA          400,000 beads 19 / 19 / 15, 39 / 29 / 29
//                             1 million   34 / 40 / 29, 75 / 60 / 54
//                             4 million   144 / 185 / 138, 295 / 270 / 230
//     with the extensile term 1 million   45 / 43 / 32, 133 / 74 / 69
//     soft spheres          400,000       29 / 35 / 21, 123 / 52 / 51
//                             1 million   54 / 80 / 43, 229 / 120 / 102
//                             4 million   208 / 368 / 199, 824 / 523 / 412
// 27 cells, one lane / 4 lanes / 2 lanes: soft spheres of 800,000 161 / 108 /
// 128, 431 / 159 / 202; WCA of 800,000 88 / 76 / 85, 158 / 98 / 119, of 4
// million 374 / 412 / 447, 687 / 543 / 656.  At 200,000 beads and below 8 lanes
// are the fastest of all in both states.
inline int pair_lanes(uint64_t beads, bool oneLayer) { return beads <= 200000u ? 8 : (oneLayer ? 2 : 4); }

}  // namespace nw
