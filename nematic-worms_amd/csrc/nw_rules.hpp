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

}  // namespace nw
