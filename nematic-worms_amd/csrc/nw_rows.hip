// nw_rows.hip -- cell order and WCA pair forces of a small system in one
// launch (gfx950).
//
// The two-level cell sort and the pair pass are three launches, each a chain
// of dependent phases on a mostly idle chip when the system has some ten
// thousand beads: 5.9 + 8.7 + 12.2 us at 32,000 beads.  Here a workgroup owns
// `rows` consecutive rows of a one-layer grid.  It reads the cell of every bead
// (a few hundred KB, from L2), keeps the beads of its rows and of the row on
// either side -- one interval of cells modulo the grid, so the wrap in y needs
// no case of its own and whole rows hold the wrap in x -- orders them in LDS
// by (cell, id), counts the beads of the rows before its own (its first sorted
// slot), writes its part of the order and evaluates its beads' pairs from LDS.
// Nothing passes between workgroups.  At 32,000 beads the launch takes 10.9 us:
// 4.3 the read of the cells (issue: some four VALU a cell in 16 wavefronts),
// 2.9 the order, 1.7 the pairs, the rest the dispatch.
//
// The pairs: four lanes a bead, lane q evaluating candidates q, q + 4, ... of
// the flattened list, their terms added in list order by quad broadcasts: the
// sums of k_collide_rows bit for bit, in a quarter of its dependent steps.
#include <algorithm>

#include "nw_bucket.hpp"
#include "nw_pair.hpp"

namespace nw {

// threads of a workgroup: 1024 read the cells of 32,000 beads in 3.4 us, 512 in
// 5.6, 256 in 10.5 (kernel 10.9 / 14.1 / 21.8 us; at 4,000 beads 6.6 / 6.8 / 7.5)
constexpr int kRowsBlock = 1024;

struct RowsArgs {
    const uint32_t *hash;  // cell of every bead, bead order
    const float4 *pos;
    float4 *force;
    uint32_t *ids, *off, *sCell;
    float4 *sPos;
};

// LDS of a workgroup (bytes): staged beads `cap`, cells of its rows and the two beside them
struct RowsLayout {
    uint32_t cnt, cur, wsum, pos, lid, lcell, total;
};
__host__ __device__ inline RowsLayout rows_layout(uint32_t cap, uint32_t cells) {
    RowsLayout L;
    uint32_t o = 0;
    L.pos = o;   o += 16u * cap;  // while the beads are collected: their groups of four
    L.lid = o;   o += 4u * cap;
    L.lcell = o; o += 2u * cap;
    o = (o + 15u) & ~15u;
    L.cnt = o;   o += 4u * (cells + 1u);
    L.cur = o;   o += 4u * cells;
    L.wsum = o;  o += 4u * 40u;
    L.total = (o + 15u) & ~15u;
    return L;
}

// the three stencil cells of x in stencil order: an inner cell's neighbours
// in one piece, an edge cell's in two (x = 0: Gx - 1, then 0 and 1; x = Gx -
// 1: Gx - 2 and Gx - 1, then 0), as [a0, a1) and [b0, b1) within a row
__device__ __forceinline__ void row_pieces(uint32_t x, uint32_t Gx, uint32_t &a0, uint32_t &a1, uint32_t &b0,
                                           uint32_t &b1) {
    const bool left = x == 0u, right = x + 1u == Gx;
    a0 = left ? Gx - 1u : x - 1u;
    a1 = left || right ? Gx : x + 2u;
    b0 = 0u;
    b1 = left ? 2u : (right ? 1u : 0u);
}

// A stage too small for the rows' beads (a collapsed or exploded system; the
// host gives it two and a half times the average): every lane takes a cell,
// then a bead, and passes over all cells of the system in bead order.  Slow
// and exact.  (LDS holds the counts of the rows' cells only.)
__device__ __forceinline__ void rows_unstaged(const KP &kp, const RowsArgs &a, uint32_t N, uint32_t idBase,
                                           uint32_t cellBase, uint32_t slotBase, uint32_t y0, uint32_t own,
                                           const uint32_t *cnt) {
    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y;
    const uint32_t first = cnt[Gx];
    for (uint32_t c = threadIdx.x; c < own * Gx; c += blockDim.x) {
        const uint32_t cell = cellBase + y0 * Gx + c;
        uint32_t w = slotBase + cnt[Gx + c] - first;
        const uint32_t e = slotBase + cnt[Gx + c + 1u] - first;
        for (uint32_t j = 0; j < N && w < e; ++j) {
            if (a.hash[j] != cell) continue;
            a.ids[w] = idBase + j;
            a.sCell[w] = cell;
            a.sPos[w] = load4(a.pos, j);
            ++w;
        }
    }
    __syncthreads();
    const float rc2 = kp.e.wcaCutoff * kp.e.wcaCutoff;
    const uint32_t beads = cnt[(own + 1u) * Gx] - first;
    for (uint32_t s = threadIdx.x; s < beads; s += blockDim.x) {
        const uint32_t me = a.ids[slotBase + s] - idBase;
        int gx, gy, gz;
        cell_xyz(kp, a.sCell[slotBase + s] - cellBase, gx, gy, gz);
        const f3 r = mk(load4(a.pos, me));
        uint32_t fil, ch;
        worm_of(kp, me, fil, ch);
        f3 acc = mk(0.f, 0.f, 0.f);
        for (int yi = -1; yi <= 1; ++yi) {
            const uint32_t y = uint32_t(gy + yi < 0 ? int(Gy) - 1 : (gy + yi == int(Gy) ? 0 : gy + yi));
            uint32_t lo, hi, b0, b1;
            row_pieces(uint32_t(gx), Gx, lo, hi, b0, b1);
            for (uint32_t k = 0; k < 3u; ++k) {
                const uint32_t cell = cellBase + y * Gx + (lo + k < hi ? lo + k : b0 + k - (hi - lo));
                for (uint32_t j = 0; j < N; ++j) {
                    if (a.hash[j] != cell) continue;
                    uint32_t fil2, ch2;
                    worm_of(kp, j, fil2, ch2);
                    float4 P = load4(a.pos, j);
                    P.w = __uint_as_float(fil2);
                    acc += wca_term_masked(kp, r, fil, rc2, P);
                }
            }
        }
        const float4 F = load4(a.force, me);
        a.force[me] = make_float4(F.x + acc.x, F.y + acc.y, F.z + acc.z, F.w + 0.0f);
    }
}

// Rows [y0, y0 + rows) of one system: N beads whose arrays hash, pos, force
// start at its first bead; ids, sCell and sPos (indexed by sorted slot) and
// off (by cell) at its own first entries; bead ids, cells and slots of the
// system are written with idBase, cellBase and slotBase added.
template <int T>
__device__ __forceinline__ void rows_body(const KP &kp, const RowsArgs &a, uint32_t N, uint32_t idBase,
                                          uint32_t cellBase, uint32_t slotAdd, uint32_t y0, uint32_t rows,
                                          uint32_t cap, uint32_t maxCells, unsigned char *smem) {
    const RowsLayout L = rows_layout(cap, maxCells);
    float4 *lpos = reinterpret_cast<float4 *>(smem + L.pos);
    uint32_t *group = reinterpret_cast<uint32_t *>(smem + L.pos);  // until the positions come: 4 cap words
    uint32_t *lid = reinterpret_cast<uint32_t *>(smem + L.lid);
    uint16_t *lcell = reinterpret_cast<uint16_t *>(smem + L.lcell);
    uint32_t *cnt = reinterpret_cast<uint32_t *>(smem + L.cnt);
    uint32_t *cur = reinterpret_cast<uint32_t *>(smem + L.cur);
    uint32_t *wsum = reinterpret_cast<uint32_t *>(smem + L.wsum);  // 16 scan sums, 16 counts below, groups

    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y, C = Gx * Gy;
    const uint32_t own = min(rows, Gy - y0);
    const uint32_t nc = (own + 2u) * Gx;                                // cells of the staged rows
    const uint32_t hOwn = y0 * Gx, hLo = (y0 == 0u ? Gy - 1u : y0 - 1u) * Gx;
    const uint32_t t = threadIdx.x;
    for (uint32_t c = t; c < nc; c += T) cnt[c] = 0u;
    if (t == 0) wsum[32] = 0u;
    __syncthreads();

    // Every bead's cell: below the own rows (counted) and, in groups of four
    // words, whether one lies in the staged rows (its local cell is the
    // distance from the first staged cell).  16-byte loads from the first
    // aligned word, eight a thread in flight; a wavefront lists its groups
    // with a staged bead by one append.  The words before the first whole
    // group are group `quads`, those after the last one quads + 1.
    // the staged cells: nA from hLo on and, past the grid's end, the first nB
    const uint32_t nA = min(nc, C - hLo), nB = nc - nA;
    auto local = [&](uint32_t h) {
        const uint32_t d = h - hLo;
        return d < nA ? d : (h < nB ? nA + h : ~0u);
    };
    const uint32_t head = min((4u - (uint32_t(reinterpret_cast<uintptr_t>(a.hash)) >> 2 & 3u)) & 3u, N);
    const uint32_t quads = (N - head) / 4u, rest = head + 4u * quads;
    const uint4 *h4 = reinterpret_cast<const uint4 *>(a.hash + head);
    uint32_t below = 0;
    // one group: whether it holds a staged bead
    auto look = [&](const uint4 &x) {
        const uint32_t h0 = x.x - cellBase, h1 = x.y - cellBase, h2 = x.z - cellBase, h3 = x.w - cellBase;
        below += h0 < hOwn ? 1u : 0u;
        below += h1 < hOwn ? 1u : 0u;
        below += h2 < hOwn ? 1u : 0u;
        below += h3 < hOwn ? 1u : 0u;
        const uint32_t d = min(min(h0 - hLo, h1 - hLo), min(h2 - hLo, h3 - hLo));
        return d < nA || min(min(h0, h1), min(h2, h3)) < nB;
    };
    // (the whole wavefront) lists the groups q + T b of the bits b of hit
    auto list = [&](uint32_t hit, uint32_t q) {
        if (!__any(hit != 0u)) return;
        const uint32_t n = uint32_t(__popc(hit)), incl = wave_scan_add(n);
        uint32_t at = 0;
        if ((t & 63u) == 63u) at = atomicAdd(&wsum[32], incl);
        at = wave_last_lane(at) + incl - n;
        for (; hit; hit &= hit - 1u, ++at)
            if (at < 4u * cap) group[at] = q + uint32_t(__builtin_ctz(hit)) * T;
    };
    constexpr uint32_t U = 8;
    const uint32_t whole = quads / T;  // rounds in which every thread has a group
    for (uint32_t r = 0; r < whole; r += U) {
        uint4 x[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (r + u < whole) x[u] = h4[(r + u) * T + t];
        uint32_t hit = 0;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (r + u < whole) hit |= look(x[u]) ? 1u << u : 0u;
        list(hit, r * T + t);
    }
    if (whole * T < quads) {
        const uint32_t q = whole * T + t;
        uint32_t hit = 0;
        if (q < quads) hit = look(h4[q]) ? 1u : 0u;
        list(hit, q);
    }
    if (t < head + (N - rest)) {
        below += a.hash[t < head ? t : rest + (t - head)] - cellBase < hOwn ? 1u : 0u;
        if (t == 0) {
            const uint32_t at = atomicAdd(&wsum[32], 2u);
            if (at < 4u * cap) group[at] = quads;
            if (at + 1u < 4u * cap) group[at + 1u] = quads + 1u;
        }
    }
    below = wave_scan_add(below);
    if ((t & 63u) == 63u) wsum[16u + (t >> 6)] = below;
    __syncthreads();
    const uint32_t slotBase = slotAdd + wave_last_lane(wave_scan_add((t & 63u) < uint32_t(T / 64) ? wsum[16u + (t & 63u)] : 0u));
    const uint32_t words = 4u * wsum[32];
    // word k of the listed groups: its bead, or N (group quads: the words
    // before the first whole group, quads + 1: those after the last)
    auto bead_of = [&](uint32_t k) {
        const uint32_t g = group[k >> 2], i = k & 3u;
        if (g < quads) return head + 4u * g + i;
        return g == quads ? (i < head ? i : N) : min(rest + i, N);
    };
    const bool listed = words <= 16u * cap;
    uint32_t id0 = N, d0 = ~0u;  // the thread's first word
    for (uint32_t k = t; k < (listed ? words : N); k += T) {
        const uint32_t id = listed ? bead_of(k) : k;
        const uint32_t d = id < N ? local(a.hash[id] - cellBase) : ~0u;
        if (d < nc) atomicAdd(&cnt[d], 1u);
        if (k == t) id0 = id, d0 = d;
    }
    __syncthreads();
    block_excl_scan<true>(cnt, nc, wsum, cur);
    const uint32_t m = cnt[nc];  // staged beads
    const uint32_t s0 = cnt[Gx], s1 = cnt[(own + 1u) * Gx];  // the own beads' staged slots
    // CSR offsets of the own cells
    for (uint32_t c = t; c < own * Gx; c += T) a.off[hOwn + c] = slotBase + cnt[Gx + c] - s0;
    if (y0 + own == Gy && t == 0) a.off[C] = slotAdd + N;
    if (m > cap) {
        rows_unstaged(kp, a, N, idBase, cellBase, slotBase - slotAdd, y0, own, cnt);
        return;
    }
    for (uint32_t k = t; k < words; k += T) {
        const uint32_t id = k == t ? id0 : bead_of(k);
        const uint32_t d = k == t ? d0 : (id < N ? local(a.hash[id] - cellBase) : ~0u);
        if (d < nc) {
            const uint32_t s = atomicAdd(&cur[d], 1u);
            lid[s] = id;
            lcell[s] = uint16_t(d);
        }
    }
    __syncthreads();
    // a cell's beads in ascending id (MD cells hold about one)
    for (uint32_t c = t; c < nc; c += T) {
        const uint32_t z = cnt[c + 1u];
        for (uint32_t u = cnt[c] + 1u; u < z; ++u) {
            const uint32_t x = lid[u];
            uint32_t w = u;
            while (w > cnt[c] && lid[w - 1u] > x) {
                lid[w] = lid[w - 1u];
                --w;
            }
            lid[w] = x;
        }
    }
    __syncthreads();
    // positions (and worm) of the staged beads; the own ones' part of the order
    for (uint32_t s = t; s < m; s += T) {
        const uint32_t id = lid[s];
        const float4 P = load4(a.pos, id);
        uint32_t fil, ch;
        worm_of(kp, id, fil, ch);
        lpos[s] = make_float4(P.x, P.y, P.z, __uint_as_float(fil));
        if (s >= s0 && s < s1) {
            const uint32_t g = slotBase - slotAdd + (s - s0);
            a.ids[g] = idBase + id;
            a.sCell[g] = cellBase + hOwn + (uint32_t(lcell[s]) - Gx);
            a.sPos[g] = P;
        }
    }
    __syncthreads();

    const float rc2 = kp.e.wcaCutoff * kp.e.wcaCutoff;
    const uint32_t lane = t & 3u;
    for (uint32_t s = s0 + t / 4u; s < s1; s += T / 4u) {
        const uint32_t me = lid[s];
        const float4 F = load4(a.force, me);
        const float4 O = lpos[s];
        const f3 r = mk(O);
        const uint32_t fil = __float_as_uint(O.w), c = lcell[s];
        const uint32_t ly = div_exact(c, kp.gxMagic, Gx), x = c - ly * Gx, row = (ly - 1u) * Gx;
        uint32_t a0, a1, b0, b1;
        row_pieces(x, Gx, a0, a1, b0, b1);
        // pieces k of slots pre[k] .. pre[k + 1] of the list, at slot t + d[k]
        uint32_t pre[7], d[6];
        pre[0] = 0u;
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            const uint32_t R = row + uint32_t(y) * Gx;
            const uint32_t p0 = cnt[R + a0], p1 = cnt[R + a1], q0 = cnt[R], q1 = cnt[R + b1];
            d[2 * y] = p0 - pre[2 * y];
            pre[2 * y + 1] = pre[2 * y] + (p1 - p0);
            d[2 * y + 1] = q0 - pre[2 * y + 1];
            pre[2 * y + 2] = pre[2 * y + 1] + (q1 - q0);
        }
        const uint32_t K = pre[6];
        f3 acc = mk(0.f, 0.f, 0.f);
        for (uint32_t i = lane; i - lane < K; i += 4u) {
            uint32_t j = d[5];
#pragma unroll
            for (int k = 4; k >= 0; --k) j = i < pre[k + 1] ? d[k] : j;
            const bool on = i < K;
            float4 P = lpos[on ? i + j : s];  // past the list: the bead itself, masked by its worm
            add_quad(acc, wca_term_masked(kp, r, fil, rc2, P));
        }
        if (lane == 0u) a.force[me] = make_float4(F.x + acc.x, F.y + acc.y, F.z + acc.z, F.w + 0.0f);
    }
}

__global__ __launch_bounds__(kRowsBlock) void k_rows(RowsArgs a, uint32_t N, uint32_t rows, uint32_t cap,
                                                     uint32_t maxCells, KP kp) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t b = xcd_contiguous(blockIdx.x, gridDim.x);
    rows_body<kRowsBlock>(kp, a, N, 0u, 0u, 0u, b * rows, rows, cap, maxCells, smem);
}

// the same of every replica of a batch: a workgroup belongs to one replica
__global__ __launch_bounds__(kRowsBlock) void k_rows_batch(BatchArrays a, const BatchRep *__restrict__ reps,
                                                           uint32_t R, uint32_t cap, uint32_t maxCells,
                                                           uint64_t *__restrict__ stepCtr) {
    extern __shared__ __align__(16) unsigned char smem[];
    // the step's last kernel advances the step counter the next front reads
    if (blockIdx.x == 0 && threadIdx.x == 0) stepCtr[0] = stepCtr[0] + 1u;
    const uint32_t b = xcd_contiguous(blockIdx.x, gridDim.x);
    const BatchRep &rep = reps[__builtin_amdgcn_readfirstlane(replica_of_row_block(reps, R, b))];
    const uint32_t b0 = rep.beadOffset, c0 = rep.cellOffset;
    const RowsArgs x{a.hash + b0,    a.pos + b0, (a.swapForces ? a.forceOld : a.force) + b0, a.ids + b0,
                     a.off + c0,     a.sCell + b0, a.sPos + b0};
    rows_body<kRowsBlock>(rep.kp, x, rep.numBeads, b0, c0, b0, (b - rep.rowBlock) * rep.rows, rep.rows, cap, maxCells,
                          smem);
}

// ---------------------------------------------------------------------------
// plan and launcher
// ---------------------------------------------------------------------------
// Every workgroup reads every bead's cell, so the launch wins while that read
// is short.  A whole step with the sort and the pair kernel / with this launch:
// 21.1 / 12.0 us at 6,400 beads, 21.5 / 15.1 at 32,000, 22.0 / 20.8 at 64,000,
// 21.3 / 22.3 at 69,000, 22.5 / 23.4 at 80,000, 23.4 / 27.5 at 112,000.
constexpr uint64_t kRowsMaxBeads = 65536;
constexpr uint32_t kRowsMaxBlocks = 256;  // one round of the CUs: 64,000 beads over 291 rows take 23.0 us by single rows, 16.0 by pairs
constexpr uint32_t kRowsMaxOwn = 768;     // beads of a workgroup on average: three rounds of its quads

// whether the launch computes a system's pair term at all
static bool rows_term(const KP &kp) {
    const SimParams &p = kp.p;
    return kp.e.pairPotential == NW_PAIR_WCA && p.activity == 0.0f && kp.e.stencil == NW_STENCIL_2D &&
           kp.e.collideKernel == NW_COLLIDE_AUTO && p.gridSize.z == 1 && p.gridSize.x >= 3 && p.gridSize.y >= 3;
}

// beads staged by a workgroup of `rows` rows: two and a half times the
// average, since rows fill to at most about the close packing of their cells
static uint32_t rows_cap(uint64_t N, uint32_t Gy, uint32_t rows) {
    return std::max(1024u, (uint32_t(2.5 * double(N) / Gy * (rows + 2u)) + 255u) & ~255u);
}

static bool rows_fits(RowsPlan &pl) {
    pl.lds = rows_layout(pl.cap, pl.cells).total;
    return pl.cells <= 8192u && pl.cap <= 8192u && pl.lds <= 150u * 1024u;
}

bool rows_plan(uint64_t N, const KP &kp, RowsPlan &out) {
    const Tuning &t = tuning();
    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y;
    if (!rows_term(kp)) return false;
    // a launch shape asked of the sort or the pair kernel is theirs
    if (t.mdTileItems || t.mdMembers || t.pairBlock || t.pairStage) return false;
    if (N == 0 || N > kRowsMaxBeads) return false;
    out.rows = std::min((Gy + kRowsMaxBlocks - 1u) / kRowsMaxBlocks, Gy - 2u);
    out.blocks = (Gy + out.rows - 1u) / out.rows;
    if (double(N) / Gy * out.rows > double(kRowsMaxOwn)) return false;
    out.cells = (out.rows + 2u) * Gx;
    out.cap = rows_cap(N, Gy, out.rows);
    return rows_fits(out);
}

// The batch takes the launch when its workgroups are done sooner than the sort
// and the pair kernel.  Measured with one size of replica throughout (us a
// step, sort + pairs / this launch): 16 x 1,100 beads 30.4 / 17.0, 16 x 8,600
// 35.5 / 24.4, 64 x 7,700 52.6 / 47.5, 64 x 4,100 43.8 / 34.2, 128 x 4,000 54.3
// / 46.4, 256 x 2,000 56.4 / 49.1, 16 x 30,000 52.3 / 48.8; the launch alone
// loses at 64 x 30,000 (95 us) and 16 x 60,000 (62).  The sort and the pairs
// take some 19 us and 26 us a million beads, 256 workgroups here 8 us and 1 us
// for every 10,000 beads of their replica.
bool rows_plan_batch(BatchRep *reps, uint32_t R, RowsPlan &out) {
    out = RowsPlan{};
    uint64_t rows = 0;
    for (uint32_t r = 0; r < R; ++r) {
        if (!rows_term(reps[r].kp)) return false;
        rows += reps[r].kp.p.gridSize.y;
    }
    RowsPlan pl{};
    const uint32_t per = uint32_t((rows + kRowsMaxBlocks - 1u) / kRowsMaxBlocks);
    double here = 0.0, beads = 0.0;
    for (uint32_t r = 0; r < R; ++r) {
        BatchRep &q = reps[r];
        const uint32_t Gx = q.kp.p.gridSize.x, Gy = q.kp.p.gridSize.y;
        const double perRow = std::max(1.0, double(q.numBeads) / Gy);
        if (perRow > double(kRowsMaxOwn)) return false;
        q.rows = std::max(1u, std::min({per, uint32_t(kRowsMaxOwn / perRow), Gy - 2u}));
        q.rowBlock = pl.blocks;
        const uint32_t blocks = (Gy + q.rows - 1u) / q.rows;
        pl.blocks += blocks;
        pl.cells = std::max(pl.cells, (q.rows + 2u) * Gx);
        pl.cap = std::max(pl.cap, rows_cap(q.numBeads, Gy, q.rows));
        here += blocks * (8.0 + 1e-4 * q.numBeads) / kRowsMaxBlocks;
        beads += q.numBeads;
    }
    if (!pl.blocks || here > 19.0 + 26e-6 * beads || !rows_fits(pl)) return false;
    out = pl;
    return true;
}

hipError_t launch_rows_batch(const RowsPlan &pl, const BatchArrays &a, const BatchRep *reps, uint32_t R,
                             uint64_t *stepCtr, hipStream_t st) {
    const hipError_t e = grant_lds(reinterpret_cast<const void *>(&k_rows_batch), pl.lds);
    if (e != hipSuccess) return e;
    NW_LAUNCH(k_rows_batch, dim3(pl.blocks), dim3(kRowsBlock), pl.lds, st, a, reps, R, pl.cap, pl.cells, stepCtr);
    return hipGetLastError();
}

hipError_t launch_rows(const RowsPlan &pl, const uint32_t *hash, const float4 *pos, float4 *force, uint32_t *ids,
                       uint32_t *off, uint32_t *sCell, float4 *sPos, uint32_t N, const KP &kp, hipStream_t st) {
    const RowsArgs a{hash, pos, force, ids, off, sCell, sPos};
    const hipError_t e = grant_lds(reinterpret_cast<const void *>(&k_rows), pl.lds);
    if (e != hipSuccess) return e;
    NW_LAUNCH(k_rows, dim3(pl.blocks), dim3(kRowsBlock), pl.lds, st, a, N, pl.rows, pl.cap, pl.cells, kp);
    return hipGetLastError();
}

}  // namespace nw
