// nw_pairs.hip -- pair forces over any stencil (gfx950): the pair pass of the
// per-call path (collideFilaments) and of fused steps whose stencil spans
// several layers of cells.
//
// In three dimensions a bead has some twenty candidates in 27 cells, and a
// system of 30,000 to 100,000 beads gives one bead per lane only one or two
// wavefronts per SIMD, each waiting on its own chain of loads.  Here S lanes
// share a bead: each looks up its share of the cells, the lanes' counts are
// scanned, and the bead's candidates are written to one LDS list, from which
// the S lanes take them in turn.  The lanes' sums are added in a fixed order.
// Measured at 96,000 beads, 64 x 64 x 32 cells: 86 -> 23.7 us against one lane a
// bead (22,600 instructions of unrolled walk, nine divisions a candidate); at
// 30,000 beads through the reference's tables 80 -> 12.5 us.  What bounds it now
// is the issue of some 950 VALU a wavefront (8 beads), exact square roots and
// quotients among them.
#include "nw_internal.hpp"
#include "nw_pair.hpp"
#include "nw_rules.hpp"

namespace nw {

// cells of the grid as runs of sorted slots: CSR offsets (cell h holds slots
// off[h] .. off[h + 1]) or the reference's tables (start 0xffffffff: empty)
struct PairCells {
    const uint32_t *off;
    const uint32_t *start, *end;
};

// A bead's candidates listed at a time (more: further rounds).  With two lanes
// a bead a workgroup holds 128 lists, and their length sets how many
// workgroups fit a CU's LDS (1 million soft spheres in one layer, in rows: 54
// us with 32 entries, 43 with 24).
constexpr uint32_t list_cap(int lanes) { return lanes <= 2 ? 24u : 64u; }

// exclusive prefix sum of v over the S lanes of a group, and its total
template <int S>
__device__ __forceinline__ uint32_t group_scan(uint32_t v, uint32_t s, uint32_t &total) {
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < S; d <<= 1) {
        const uint32_t y = __shfl_up(x, d, S);
        x += s >= uint32_t(d) ? y : 0u;
    }
    total = __shfl(x, S - 1, S);
    return x - v;
}

// CELLS: the stencil's cells, 9 of one layer or 27
template <int MODE, bool TAN, bool UNIT, bool CSR, int S, int CELLS>
__global__ __launch_bounds__(kBlock) void k_pair_list(float4 *__restrict__ force, const float4 *__restrict__ sPos,
                                                      const float4 *__restrict__ sVel,
                                                      const float4 *__restrict__ sTan,
                                                      const uint32_t *__restrict__ sIdx, PairCells cells,
                                                      const uint32_t *__restrict__ sCell, uint32_t n, KP kp) {
    constexpr uint32_t G = kBlock / S;           // beads of a workgroup
    constexpr uint32_t kListCap = list_cap(S);
    constexpr uint32_t PER = (CELLS + S - 1) / S;  // cells of a lane
    __shared__ uint32_t list[G][kListCap];
    __shared__ float listW[UNIT ? 1 : G][UNIT ? 1 : kListCap];
    const SimParams &p = kp.p;
    const uint32_t g = threadIdx.x / S, s = threadIdx.x % S;
    // neighbouring workgroups share cells: contiguous runs of them per XCD
    const uint32_t i = xcd_contiguous(blockIdx.x, gridDim.x) * G + g;
    const bool own = i < n;
    const uint32_t ic = own ? i : n - 1u;  // groups past the end take the last bead, unused
    const uint32_t me = sIdx[ic];
    const Owner<MODE, TAN> o = load_owner<MODE, TAN>(kp, ic, me, sPos, sVel, sTan);
    int gx, gy, gz;
    if (CSR) {
        cell_xyz(kp, sCell[ic], gx, gy, gz);
    } else {
        gx = wrap_mod(cell_coord(o.r.x, p.origin.x, p.cellSize.x), p.gridSize.x);
        gy = wrap_mod(cell_coord(o.r.y, p.origin.y, p.cellSize.y), p.gridSize.y);
        gz = wrap_mod(cell_coord(o.r.z, p.origin.z, p.cellSize.z), p.gridSize.z);
    }
    const AxisCells ax = axis_cells_in(gx, p.gridSize.x, false);
    const AxisCells ay = axis_cells_in(gy, p.gridSize.y, false);
    const AxisCells az = axis_cells_in(gz, p.gridSize.z, kp.e.stencil == NW_STENCIL_2D);

    // The lane's cells, PER in a row of them (x fastest, so the list runs
    // through the sorted slots row by row); one beyond an
    // axis's distinct cells counts nothing.  Every load is unconditional and
    // in bounds (an unused entry of AxisCells holds the centre).
    uint32_t a[PER], end[PER], len[PER], total = 0;
    bool use[PER];
    float wt[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t k = s * PER + j, kc = min(k, uint32_t(CELLS) - 1u);
        const uint32_t zi = CELLS == 9 ? 0u : kc / 9u, yi = kc / 3u % 3u, xi = kc % 3u;
        const int cx = xi == 0 ? ax.c[0] : (xi == 1 ? ax.c[1] : ax.c[2]);
        const int cy = yi == 0 ? ay.c[0] : (yi == 1 ? ay.c[1] : ay.c[2]);
        const int cz = zi == 0 ? az.c[0] : (zi == 1 ? az.c[1] : az.c[2]);
        const uint32_t h = (uint32_t(cz) * p.gridSize.y + uint32_t(cy)) * p.gridSize.x + uint32_t(cx);
        use[j] = own && k < uint32_t(CELLS) && int(xi) < ax.n && int(yi) < ay.n && int(zi) < az.n;
        // (an empty cell's entry of `end` holds what it held, unused)
        a[j] = CSR ? cells.off[h] : cells.start[h];
        end[j] = CSR ? cells.off[h + 1u] : cells.end[h];
        if (!UNIT) {
            wt[j] = (zi == 0 ? az.w[0] : (zi == 1 ? az.w[1] : az.w[2])) *
                    (yi == 0 ? ay.w[0] : (yi == 1 ? ay.w[1] : ay.w[2])) *
                    (xi == 0 ? ax.w[0] : (xi == 1 ? ax.w[1] : ax.w[2]));
        }
    }
    // the ends loaded beside the starts, not behind a branch on each (30,000
    // beads by the tables: 14.4 us with it, 12.8 without)
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) asm volatile("" ::"v"(end[j]));
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const bool any = use[j] && (CSR || a[j] != 0xffffffffu);
        len[j] = any && end[j] > a[j] ? end[j] - a[j] : 0u;
        total += len[j];
    }
    uint32_t K;
    const uint32_t first = group_scan<S>(total, s, K);

    const float rc2 = kp.e.wcaCutoff * kp.e.wcaCutoff;
    f3 acc = mk(0.f, 0.f, 0.f);
    // a wavefront's groups list and take their candidates together; the
    // lists belong to the wavefront, whose lanes run in step
    for (uint32_t base = 0; __any(base < K); base += kListCap) {
        // of each cell the entries of this round alone: a cell crowded beyond
        // the list is listed once over all rounds, not once in each
        uint32_t f = first;
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            const uint32_t k0 = f < base ? min(base - f, len[j]) : 0u;
            const uint32_t k1 = f < base + kListCap ? min(base + kListCap - f, len[j]) : 0u;
#pragma unroll 1
            for (uint32_t k = k0; k < k1; ++k) {
                list[g][f + k - base] = a[j] + k;
                if (!UNIT) listW[g][f + k - base] = wt[j];
            }
            f += len[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t m = K > base ? min(K - base, kListCap) : 0u;
        for (uint32_t t = s; t < m; t += S) {
            const uint32_t j0 = list[g][t];
            const uint32_t I0 = sIdx[j0];
            const float4 P0 = load4(sPos, j0);
            float4 V0{}, T0{};
            if (MODE == 0) V0 = load4(sVel, j0);
            if (TAN) T0 = load4(sTan, j0);
            // by the bead ids alone: the owner's worm starts at me - o.ch
            const bool same = I0 - (me - o.ch) < p.filamentSize;
            const PairWho who{I0 == me, same, same && (I0 + 1u == me || I0 - 1u == me)};
            add_pair<MODE, TAN, UNIT>(kp, o, rc2, UNIT ? 1.0f : listW[g][t], acc, mk(P0), who, mk(V0), mk(T0));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // the lanes' sums in a fixed tree
#pragma unroll
    for (int d = S / 2; d >= 1; d >>= 1)
        acc += mk(__shfl_down(acc.x, d, S), __shfl_down(acc.y, d, S), __shfl_down(acc.z, d, S));
    if (own && s == 0u) {
        const float4 F = load4(force, me);
        force[me] = make_float4(F.x + acc.x, F.y + acc.y, F.z + acc.z, F.w + 0.0f);
    }
}

template <bool CSR, int S, int CELLS>
static void launch_list_of(float4 *force, const float4 *sPos, const float4 *sVel, const float4 *sTan,
                           const uint32_t *sIdx, const PairCells &c, const uint32_t *sCell, uint32_t n, const KP &kp,
                           hipStream_t st) {
    const bool wca = kp.e.pairPotential == NW_PAIR_WCA;
    const bool tan = !wca || kp.p.activity != 0.0f;
    // every distinct cell counts once when no axis folds its offsets
    const bool unit = kp.p.gridSize.x >= 3 && kp.p.gridSize.y >= 3 &&
                      (kp.e.stencil == NW_STENCIL_2D || kp.p.gridSize.z >= 3);
    const dim3 grid(grid_for(uint64_t(n) * S)), block(kBlock);
#define NW_LIST(M, T, U) \
    NW_LAUNCH((k_pair_list<M, T, U, CSR, S, CELLS>), grid, block, 0, st, force, sPos, sVel, sTan, sIdx, c, sCell, n, kp)
    if (unit) {
        if (!wca) NW_LIST(0, true, true);
        else if (tan) NW_LIST(1, true, true);
        else NW_LIST(1, false, true);
    } else {
        if (!wca) NW_LIST(0, true, false);
        else if (tan) NW_LIST(1, true, false);
        else NW_LIST(1, false, false);
    }
#undef NW_LIST
}

template <bool CSR>
static hipError_t launch_list(float4 *force, const float4 *sPos, const float4 *sVel, const float4 *sTan,
                              const uint32_t *sIdx, const PairCells &c, const uint32_t *sCell, uint32_t n,
                              const KP &kp, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const bool oneLayer = kp.e.stencil == NW_STENCIL_2D || kp.p.gridSize.z == 1;
    const int lanes = pair_lanes(n, oneLayer);
#define NW_LIST_OF(S, CELLS) launch_list_of<CSR, S, CELLS>(force, sPos, sVel, sTan, sIdx, c, sCell, n, kp, st)
    if (oneLayer) {
        if (lanes == 8) NW_LIST_OF(8, 9);
        else NW_LIST_OF(2, 9);
    } else {
        if (lanes == 8) NW_LIST_OF(8, 27);
        else NW_LIST_OF(4, 27);
    }
#undef NW_LIST_OF
    return hipGetLastError();
}

hipError_t launch_collide_filaments(float4 *force, const float4 *sPos, const float4 *sVel, const float4 *sTan,
                                    const uint32_t *sIdx, const uint32_t *cellStart, const uint32_t *cellEnd,
                                    uint32_t n, const KP &kp, hipStream_t st) {
    return launch_list<false>(force, sPos, sVel, sTan, sIdx, PairCells{nullptr, cellStart, cellEnd}, nullptr, n, kp,
                              st);
}

hipError_t launch_collide_layers(float4 *force, const float4 *sPos, const float4 *sVel, const float4 *sTan,
                                 const uint32_t *sIdx, const uint32_t *off, const uint32_t *sCell, uint32_t n,
                                 const KP &kp, hipStream_t st) {
    return launch_list<true>(force, sPos, sVel, sTan, sIdx, PairCells{off, nullptr, nullptr}, sCell, n, kp, st);
}

}  // namespace nw
