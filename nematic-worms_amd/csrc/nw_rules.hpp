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

// The SRD sort's second level (k_srd_cells): the sorting network of a cell, 16
// or 32 ids.  A cell beyond its network is sorted by insertion, so above some
// seven particles a cell the larger one pays: in cell order a million
// particles of ten a cell 55 -> 38 us a collision, at random 55 -> 52.  But it
// holds four workgroups a CU against eight.
// With one round of it (1,024 buckets) up to some 26 a cell (500,000 of 24 86 /
// 94 us in cell order, 64 / 68 at random, of 30 118 / 117 and 76 / 75).
// Between that and one round of the smaller (2,048) it takes two: 1.1 million
// of eight at random 67 against 60 (in cell order, which the host cannot tell,
// it would still win, 50 against 56).  Beyond, where both take several, from
// ten (6 million of eight 362 / 358 at random and 193 / 182 in cell order, of
// ten 305 / 309 and 162 / 163, of twelve 352 / 358 and 208 / 222) to twenty
// (282 / 298 and 213 / 246; of 24 293 / 272 and 285 / 260).  In dense cells
// insertion is most of the work by either and what counts is how many
// workgroups wait together: 3 million of 40 a cell 443 against 324 us.
inline int srd_network(uint64_t particles, uint64_t cells, uint64_t buckets) {
    uint64_t from = 7, to = 26;  // a cell, from not included
    if (buckets > 1024u) from = 9, to = buckets > 2048u ? 21 : 0;
    return particles > from * cells && particles <= to * cells ? 32 : 16;
}

// Whether its members take their places in a pass of their own behind the
// scan, in step, instead of with their counts as their loads arrive: the ids
// of a cell then lie nearly in order, which insertion is the faster for (3
// million of 40 a cell at random 223 -> 165 us); up to twelve a cell, where the
// networks sort, one pass of atomics less is 1 % (6 million of ten in cell
// order 163 against 166).
inline bool srd_late(uint64_t particles, uint64_t cells) { return particles > 12u * cells; }

}  // namespace nw
