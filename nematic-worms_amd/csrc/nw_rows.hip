// nw_rows.hip -- cell order and WCA pair forces of a small system in one
// launch (gfx950).
//
// The two-level cell sort and the pair pass are three launches, each a chain
// of dependent phases on a mostly idle chip when the system has some ten
// thousand beads: 5.9 + 8.7 + 12.2 us at 32,000 beads.  Here a workgroup owns
// `rows` consecutive rows of a one-layer grid.  It reads the rows of cells that
// every worm spans (one word a worm, left by the front), lists the worms that
// may have a bead in its rows or in the row on either side and keeps those
// beads -- one interval of cells modulo the grid, so the wrap in y needs
// no case of its own and whole rows hold the wrap in x -- orders them in LDS
// by (cell, id), counts the beads of the rows before its own (its first sorted
// slot), writes its part of the order and evaluates its beads' pairs from LDS.
// Nothing passes between workgroups.  At 32,000 beads the launch takes 8.5 us
// (11.7 reading every bead's cell): 1.3 the worms, 2 the order, 1.5 the pairs,
// the rest the dispatch and barriers.
//
// The pairs: up to some 400 own beads four lanes a bead, lane q evaluating
// candidates q, q + 4, ... of the flattened list, their terms added in list
// order by quad broadcasts: a quarter of the dependent steps.  With more beads
// a workgroup has chains enough and a bead takes one lane (kRowsLaneBeads).
// Either way the sums of k_collide_rows bit for bit.
#include <algorithm>

#include "nw_bucket.hpp"
#include "nw_pair.hpp"
#include "nw_rules.hpp"

namespace nw {

// threads of a workgroup: 1024 against 512 and 256, 32,000 beads 10.9 / 14.1 / 21.8
// us and 4,000 6.6 / 6.8 / 7.5 (as measured with every bead's cell read)
constexpr int kRowsBlock = 1024;

struct RowsArgs {
    const uint32_t *hash;   // cell of every bead, bead order
    uint32_t *worms;        // rows of every worm (worm_rows_word); behind a system's words is its scratch
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
    L.pos = o;   o += 16u * cap;  // while the beads are collected: their worms
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

// own beads above which a bead takes one lane instead of four: 229,000 beads
// (1,140 a workgroup) 19.1 -> 16.2 us, 192,000 (770) 16.5 -> 14.7, 16 replicas of
// 8,600 (570) 12.9 -> 10.6; 64,000 (440) 11.6 -> 11.0
constexpr uint32_t kRowsLaneBeads = 400;

// The pair forces of the staged beads s0 .. s1, LANES (1 or 4) lanes a bead:
// lane q evaluates candidates q, q + LANES, ... of the flattened list, the
// terms added in list order either way.  Four lanes shorten a bead's chain,
// one costs half the instructions a candidate.
template <int T, int LANES>
__device__ __forceinline__ void rows_pairs(const KP &kp, const RowsArgs &a, const uint32_t *lid, const float4 *lpos,
                                           const uint16_t *lcell, const uint32_t *cnt, uint32_t s0, uint32_t s1) {
    const uint32_t Gx = kp.p.gridSize.x, t = threadIdx.x, lane = t % LANES;
    const float rc2 = kp.e.wcaCutoff * kp.e.wcaCutoff;
    for (uint32_t s = s0 + t / LANES; s < s1; s += T / LANES) {
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
        if (LANES == 1) {
            // without an edge bead in the wavefront every second piece is empty
            if (__any(b1 != 0u)) {
                for (uint32_t i = 0; i < K; ++i) {
                    uint32_t j = d[5];
#pragma unroll
                    for (int k = 4; k >= 0; --k) j = i < pre[k + 1] ? d[k] : j;
                    acc += wca_term_masked(kp, r, fil, rc2, lpos[i + j]);
                }
            } else {
                for (uint32_t i = 0; i < K; ++i) {
                    const uint32_t j = i < pre[1] ? d[0] : (i < pre[3] ? d[2] : d[4]);
                    acc += wca_term_masked(kp, r, fil, rc2, lpos[i + j]);
                }
            }
        } else {
            for (uint32_t i = lane; i - lane < K; i += 4u) {
                uint32_t j = d[5];
#pragma unroll
                for (int k = 4; k >= 0; --k) j = i < pre[k + 1] ? d[k] : j;
                const bool on = i < K;
                // past the list: the bead itself, masked by its worm
                add_quad(acc, wca_term_masked(kp, r, fil, rc2, lpos[on ? i + j : s]));
            }
        }
        if (lane == 0u) a.force[me] = make_float4(F.x + acc.x, F.y + acc.y, F.z + acc.z, F.w + 0.0f);
    }
}

// The scratch behind the words of a launch's worms (n beads in all): the beads
// of crowded rows beside a workgroup's own, two roles a row, as they arrive
// and in order.
struct RowsSpill {
    uint32_t *raw;  // 2 n ids
    float4 *pos;    // 2 n records: position, worm
    uint64_t n;
};
__device__ __forceinline__ RowsSpill rows_spill(uint32_t *worms, uint64_t n) {
    return {worms + n, reinterpret_cast<float4 *>(worms + ((3u * n + 3u) & ~uint64_t(3))), n};
}

// More beads than the stage holds (worms crowded into a few rows): the staged
// beads' lists in memory.  The own ones stand at their slots, as they arrive in
// sCell and in ascending id per cell in ids and sPos; those of the rows below
// and above in the spill, at the slots that their rows have in the system
// (at: its first bead): a row is below the rows of one workgroup alone, and above those of
// one, so no two workgroups meet there.
// A bead counts its own rank among the ids of its cell, so a cell takes the
// square of its beads over the threads, not one thread's insertion sort (a
// system collapsed into few cells); and it goes to its place as the record
// that the walk reads, one load a candidate.  Twelve rows of 5,000 beads: a step
// 0.57 ms, by the sort and the pair kernel 0.27, by passes over all beads 320;
// 4,000 beads in a cell or two 4.4 ms, by insertion 395; 250,000 beads in four
// tenths of their box 118 us, before the launch 101.  What bounds it is that
// the crowded rows' few workgroups do all the work.
template <typename BeadOf, typename Local>
__device__ __forceinline__ void rows_in_memory(const KP &kp, const RowsArgs &a, const RowsSpill &sp, uint32_t at,
                                               uint32_t N, uint32_t idBase, uint32_t cellBase, uint32_t slot0,
                                               uint32_t y0, uint32_t own, const uint32_t *cnt, uint32_t *cur,
                                               uint32_t words, const BeadOf &bead_of, const Local &local) {
    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y, nc = (own + 2u) * Gx;
    const uint32_t s0 = cnt[Gx], s1 = cnt[(own + 1u) * Gx], m = cnt[nc];
    // of a staged slot u: below u < s0, own, above u >= s1; its place in the spill
    const uint64_t lo = at + (y0 == 0u ? N - s0 : slot0 - s0);
    const uint64_t hi = sp.n + at + (y0 + own == Gy ? 0u : slot0 + (s1 - s0));
    auto raw = [&](uint32_t u) {
        return u < s0 ? sp.raw + lo + u : (u < s1 ? a.sCell + slot0 + (u - s0) : sp.raw + hi + (u - s1));
    };
    for (uint32_t k = threadIdx.x; k < words; k += blockDim.x) {
        const uint32_t id = bead_of(k), d = local(a.hash[id] - cellBase);
        if (d < nc) *raw(atomicAdd(&cur[d], 1u)) = id;
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < m; s += blockDim.x) {
        const uint32_t id = *raw(s), d = local(a.hash[id] - cellBase);
        const float4 P = load4(a.pos, id);
        const uint32_t c0 = cnt[d], z = cnt[d + 1u] - c0;
        const uint32_t *cell = raw(c0);
        uint32_t r = c0;
#pragma unroll 4
        for (uint32_t u = 0; u < z; ++u) r += cell[u] < id ? 1u : 0u;
        if (s >= s0 && s < s1) {
            a.ids[slot0 + (r - s0)] = idBase + id;
            a.sPos[slot0 + (r - s0)] = P;
        } else {
            uint32_t fil, ch;
            worm_of(kp, id, fil, ch);
            sp.pos[s < s0 ? lo + r : hi + (r - s1)] = make_float4(P.x, P.y, P.z, __uint_as_float(fil));
        }
    }
    __syncthreads();
    const float rc2 = kp.e.wcaCutoff * kp.e.wcaCutoff;
    for (uint32_t s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
        const uint32_t me = a.ids[slot0 + (s - s0)] - idBase, cell = a.hash[me];
        a.sCell[slot0 + (s - s0)] = cell;
        int gx, gy, gz;
        cell_xyz(kp, cell - cellBase, gx, gy, gz);
        const f3 r = mk(load4(a.sPos, slot0 + (s - s0)));
        uint32_t fil, ch, x0, x1, b0, b1;
        worm_of(kp, me, fil, ch);
        row_pieces(uint32_t(gx), Gx, x0, x1, b0, b1);
        f3 acc = mk(0.f, 0.f, 0.f);
        for (uint32_t yi = 0; yi < 3u; ++yi) {
            const uint32_t y = uint32_t(gy) - y0 + yi, row = y * Gx;  // staged: the one below the own rows first
            const bool mine = y >= 1u && y <= own;
            const float4 *rec = mine ? a.sPos + slot0 - s0 : sp.pos + (y == 0u ? lo : hi - s1);
            // the row's three cells in one run, or in two across the wrap
            for (uint32_t k = 0; k < 2u; ++k) {
                const uint32_t z = cnt[row + (k ? b1 : x1)];
#pragma unroll 2
                for (uint32_t u = cnt[row + (k ? b0 : x0)]; u < z; ++u) {
                    float4 P = load4(rec, u);
                    if (mine) {
                        uint32_t fil2, ch2;
                        worm_of(kp, a.ids[slot0 + (u - s0)] - idBase, fil2, ch2);
                        P.w = __uint_as_float(fil2);
                    }
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
// system are written with idBase, cellBase and slotBase added.  spill(): the
// launch's scratch (an argument of the launch more took 0.1 us: it has its
// place behind the worms' words).
template <int T, typename Spill>
__device__ __forceinline__ void rows_body(const KP &kp, const RowsArgs &a, uint32_t N, uint32_t idBase,
                                          uint32_t cellBase, uint32_t slotAdd, uint32_t y0, uint32_t rows,
                                          uint32_t cap, uint32_t maxCells, unsigned char *smem, const Spill &spill) {
    const RowsLayout L = rows_layout(cap, maxCells);
    float4 *lpos = reinterpret_cast<float4 *>(smem + L.pos);
    uint32_t *list = reinterpret_cast<uint32_t *>(smem + L.pos);  // until the positions come: 4 cap words
    uint32_t *lid = reinterpret_cast<uint32_t *>(smem + L.lid);
    uint16_t *lcell = reinterpret_cast<uint16_t *>(smem + L.lcell);
    uint32_t *cnt = reinterpret_cast<uint32_t *>(smem + L.cnt);
    uint32_t *cur = reinterpret_cast<uint32_t *>(smem + L.cur);
    uint32_t *wsum = reinterpret_cast<uint32_t *>(smem + L.wsum);  // 16 scan sums, 16 counts below, worms

    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y, C = Gx * Gy;
    const uint32_t own = min(rows, Gy - y0);
    const uint32_t nc = (own + 2u) * Gx;                                // cells of the staged rows
    const uint32_t hOwn = y0 * Gx, hLo = (y0 == 0u ? Gy - 1u : y0 - 1u) * Gx;
    const uint32_t t = threadIdx.x;
    for (uint32_t c = t; c < nc; c += T) cnt[c] = 0u;
    if (t == 0) wsum[32] = 0u;
    __syncthreads();

    // Every worm's rows, which the front left: a worm wholly below the own rows
    // has all its beads counted there, one that may have a bead in the staged
    // rows is listed (a wavefront's by one append), any other is passed over.
    // The own rows' first row lies between two staged ones, or is the grid's
    // first with no row below: a worm on both sides of it is listed.
    const uint32_t n = kp.p.filamentSize, W = div_exact(N, kp.fdivMagic, n);
    const uint32_t yLo = y0 == 0u ? Gy - 1u : y0 - 1u;
    const uint32_t rA = min(own + 2u, Gy - yLo), rB = own + 2u - rA;  // staged: rA rows from yLo on, the first rB
    uint32_t below = 0;
    auto look = [&](uint32_t w, uint32_t x) {
        const uint32_t lo = 0xffffu - (x >> 16), hi = x & 0xffffu;
        const bool hit = w < W && ((hi >= yLo && lo < yLo + rA) || lo < rB);
        below += w < W && !hit && hi < y0 ? n : 0u;
        const uint64_t hits = __ballot(hit);
        if (hits) {
            uint32_t at = 0;
            if ((t & 63u) == 0u) at = atomicAdd(&wsum[32], uint32_t(__popcll(hits)));
            at = __builtin_amdgcn_readfirstlane(at) +
                 __builtin_amdgcn_mbcnt_hi(uint32_t(hits >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(hits), 0u));
            if (hit && at < 4u * cap) list[at] = w;
        }
    };
    constexpr uint32_t U = 8;  // a thread's worms in flight together
    for (uint32_t w0 = 0; w0 < W; w0 += U * T) {
        uint32_t x[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (w0 + u * T < W) x[u] = a.worms[min(w0 + u * T + t, W - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (w0 + u * T < W) look(w0 + u * T + t, x[u]);
    }
    __syncthreads();
    // the cells of the listed worms' beads (of every bead when the list is too
    // short), the first kWords a thread held from here to the placement
    const uint32_t nA = min(nc, C - hLo), nB = nc - nA;
    auto local = [&](uint32_t h) {  // the distance from the first staged cell
        const uint32_t d = h - hLo;
        return d < nA ? d : (h < nB ? nA + h : ~0u);
    };
    const bool listed = wsum[32] <= 4u * cap;
    const uint32_t words = listed ? wsum[32] * n : N;
    auto bead_of = [&](uint32_t k) {
        uint32_t w, q;
        worm_of(kp, k, w, q);
        return listed ? list[w] * n + q : k;
    };
    if (!listed) below = 0u;
    constexpr uint32_t kWords = 4;
    uint32_t idk[kWords], hk[kWords];
#pragma unroll
    for (uint32_t j = 0; j < kWords; ++j) {
        const uint32_t k = t + j * T;
        idk[j] = k < words ? bead_of(k) : N;
        hk[j] = idk[j] < N ? a.hash[idk[j]] - cellBase : ~0u;
    }
    auto count = [&](uint32_t h, bool on) {
        below += on && h < hOwn ? 1u : 0u;
        const uint32_t d = on ? local(h) : ~0u;
        if (d < nc) atomicAdd(&cnt[d], 1u);
        return d;
    };
#pragma unroll
    for (uint32_t j = 0; j < kWords; ++j) hk[j] = count(hk[j], idk[j] < N);
    for (uint32_t k = t + kWords * T; k < words; k += T) (void)count(a.hash[bead_of(k)] - cellBase, true);
    below = wave_scan_add(below);
    if ((t & 63u) == 63u) wsum[16u + (t >> 6)] = below;
    __syncthreads();
    block_excl_scan<true>(cnt, nc, wsum, cur);
    const uint32_t slotBase = slotAdd + wave_last_lane(wave_scan_add((t & 63u) < uint32_t(T / 64) ? wsum[16u + (t & 63u)] : 0u));
    const uint32_t m = cnt[nc];  // staged beads
    const uint32_t s0 = cnt[Gx], s1 = cnt[(own + 1u) * Gx];  // the own beads' staged slots
    // CSR offsets of the own cells
    for (uint32_t c = t; c < own * Gx; c += T) a.off[hOwn + c] = slotBase + cnt[Gx + c] - s0;
    if (y0 + own == Gy && t == 0) a.off[C] = slotAdd + N;
    if (m > cap) {
        rows_in_memory(kp, a, spill(), slotAdd, N, idBase, cellBase, slotBase - slotAdd, y0, own, cnt, cur, words, bead_of, local);
        return;
    }
    auto place = [&](uint32_t id, uint32_t d) {
        if (d < nc) {
            const uint32_t s = atomicAdd(&cur[d], 1u);
            lid[s] = id;
            lcell[s] = uint16_t(d);
        }
    };
#pragma unroll
    for (uint32_t j = 0; j < kWords; ++j) place(idk[j], hk[j]);
    for (uint32_t k = t + kWords * T; k < words; k += T) {
        const uint32_t id = bead_of(k);
        place(id, local(a.hash[id] - cellBase));
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

    if (s1 - s0 > kRowsLaneBeads) rows_pairs<T, 1>(kp, a, lid, lpos, lcell, cnt, s0, s1);
    else rows_pairs<T, 4>(kp, a, lid, lpos, lcell, cnt, s0, s1);
}

__global__ __launch_bounds__(kRowsBlock) void k_rows(RowsArgs a, uint32_t N, uint32_t rows, uint32_t cap,
                                                     uint32_t maxCells, KP kp) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t b = xcd_contiguous(blockIdx.x, gridDim.x);
    rows_body<kRowsBlock>(kp, a, N, 0u, 0u, 0u, b * rows, rows, cap, maxCells, smem, [&] { return rows_spill(a.worms, N); });
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
    const RowsArgs x{a.hash + b0, a.wormRows + b0, a.pos + b0, (a.swapForces ? a.forceOld : a.force) + b0, a.ids + b0,
                     a.off + c0,     a.sCell + b0, a.sPos + b0};
    rows_body<kRowsBlock>(rep.kp, x, rep.numBeads, b0, c0, b0, (b - rep.rowBlock) * rep.rows, rep.rows, cap, maxCells,
                          smem, [&] {
                              const BatchRep &last = reps[R - 1u];
                              return rows_spill(a.wormRows, last.beadOffset + last.numBeads);
                          });
}

// ---------------------------------------------------------------------------
// plan and launcher
// ---------------------------------------------------------------------------
// A step with the sort and the pair kernel / with this launch, worms of 16: 21.5
// / 13.0 us at 32,000 beads, 22.1 / 16.0 at 64,000, 25.0 / 19.9 at 128,000, 27.7
// / 22.6 at 192,000, 28.9 / 27.5 at 256,000, 33.1 / 33.6 at 288,000; worms of
// 23, whose front and first sort level are two launches (front_tiles_plan: more
// than 4,096 wavefronts, as any system beyond 262,144 beads has): 32.9 / 27.9 at
// 229,000, 35.8 / 31.4 at 298,000, 39.0 / 38.8 at 344,000.
constexpr uint64_t kRowsMaxBeads = 300000;
// every workgroup reads every worm's rows: 22.8 / 20.4 us with 20,000 worms of
// three, 23.1 / 24.8 with 30,000; of five 22.7 / 19.6 with 15,000, 26.9 / 28.1
// with 30,000
constexpr uint64_t kRowsMaxWorms = 24576;
constexpr uint32_t kRowsMaxBlocks = 256;  // one round of the CUs: 64,000 beads over 291 rows take 23.0 us by single rows, 16.0 by pairs
constexpr uint32_t kRowsMaxOwn = 1408;    // beads of a workgroup on average, which its stage and its rounds allow

// whether the launch computes a system's pair term at all
static bool rows_term(const KP &kp) {
    const SimParams &p = kp.p;
    return kp.e.pairPotential == NW_PAIR_WCA && p.activity == 0.0f && kp.e.stencil == NW_STENCIL_2D &&
           kp.e.collideKernel == NW_COLLIDE_AUTO && p.gridSize.z == 1 && p.gridSize.x >= 3 && p.gridSize.y >= 3 &&
           p.gridSize.y < 65536u;  // a row in 16 bits
}

// Beads staged by a workgroup of `rows` rows: two and a half times the
// average, and as far as `lds` bytes hold them the packing of the rows' cells:
// worms that gather in bands, or start on a lattice in a part of the box, stay
// within the stage (200,000 beads in four tenths of their box, 1.75 a cell: a
// step 75 us, with the packing of single beads, 1.45 a cell, 133).
static uint32_t rows_cap(uint64_t N, const KP &kp, uint32_t rows, uint32_t lds) {
    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y;
    const uint32_t cells = (rows + 2u) * Gx, fixed = rows_layout(0, cells).total;
    const uint32_t mean = (uint32_t(2.5 * double(N) / Gy * (rows + 2u)) + 255u) & ~255u;
    const double perCell = worms_packed(double(kp.p.cellSize.x) * kp.p.cellSize.y, kp.e.wcaSigma,
                                        kp.p.filamentSize > 1 ? kp.p.bondSpringL : kp.e.wcaSigma);
    const uint32_t packed = (uint32_t(perCell * cells) + 255u) & ~255u;
    const uint32_t room = lds > fixed ? std::min((lds - fixed) / 22u & ~255u, 8192u) : 0u;
    return std::max({1024u, mean, std::min(packed, room)});
}

// LDS of a workgroup alone on its CU, and where two share one (batches, whose
// workgroups may be more than a round)
constexpr uint32_t kRowsLds = 150u * 1024u, kRowsLdsHalf = 80u * 1024u;

static bool rows_fits(RowsPlan &pl) {
    pl.lds = rows_layout(pl.cap, pl.cells).total;
    return pl.cells <= 8192u && pl.cap <= 8192u && pl.lds <= kRowsLds;
}

bool rows_plan(uint64_t N, const KP &kp, RowsPlan &out) {
    const Tuning &t = tuning();
    const uint32_t Gx = kp.p.gridSize.x, Gy = kp.p.gridSize.y;
    if (!rows_term(kp)) return false;
    // a launch shape asked of the sort or the pair kernel is theirs
    if (t.mdTileItems || t.mdMembers || t.pairBlock || t.pairStage) return false;
    if (N == 0 || N / kp.p.filamentSize > kRowsMaxWorms || N > kRowsMaxBeads) return false;
    out.rows = std::min((Gy + kRowsMaxBlocks - 1u) / kRowsMaxBlocks, Gy - 2u);
    out.blocks = (Gy + out.rows - 1u) / out.rows;
    if (double(N) / Gy * out.rows > double(kRowsMaxOwn)) return false;
    out.cells = (out.rows + 2u) * Gx;
    out.cap = rows_cap(N, kp, out.rows, kRowsLds);
    return rows_fits(out);
}

// The batch takes the launch up to 700,000 beads in replicas of up to 100,000.  A
// step (us, sort + pairs / this launch): 16 x 1,100 beads 27.8 / 13.5, 48 x 8,100
// 46 / 40, 64 x 7,700 51 / 44, 80 x 8,500 59 / 55, 16 x 29,700 49 / 44, 8 x 79,500 55
// / 50, 128 x 4,000 53 / 44, 256 x 2,000 55 / 49; past it 128 x 8,100 76 / 75, 6 x
// 127,000 57 / 61, 2 x 180,000 39 / 42.
constexpr uint64_t kRowsMaxBatchBeads = 700000, kRowsMaxReplicaBeads = 100000;

bool rows_plan_batch(BatchRep *reps, uint32_t R, RowsPlan &out) {
    out = RowsPlan{};
    uint64_t rows = 0, beads = 0;
    for (uint32_t r = 0; r < R; ++r) {
        if (!rows_term(reps[r].kp)) return false;
        rows += reps[r].kp.p.gridSize.y;
        beads += reps[r].numBeads;
    }
    RowsPlan pl{};
    const uint32_t per = uint32_t((rows + kRowsMaxBlocks - 1u) / kRowsMaxBlocks);
    // beads of a workgroup: somewhat more than an even share of a round of the
    // CUs, so that a replica denser than the rest is cut finer (16 of 800 to
    // 24,000 beads: 576 us a pass with 1,408 throughout, 565 with its 768)
    const double own = std::min(std::max(1.25 * double(beads) / kRowsMaxBlocks, 768.0), double(kRowsMaxOwn));
    for (uint32_t r = 0; r < R; ++r) {
        BatchRep &q = reps[r];
        const uint32_t Gx = q.kp.p.gridSize.x, Gy = q.kp.p.gridSize.y;
        const double perRow = std::max(1.0, double(q.numBeads) / Gy);
        if (perRow > own || q.numBeads > kRowsMaxReplicaBeads || q.kp.p.numFilaments > kRowsMaxWorms)
            return false;
        q.rows = std::max(1u, std::min({per, uint32_t(own / perRow), Gy - 2u}));
        q.rowBlock = pl.blocks;
        const uint32_t blocks = (Gy + q.rows - 1u) / q.rows;
        pl.blocks += blocks;
        pl.cells = std::max(pl.cells, (q.rows + 2u) * Gx);
        pl.cap = std::max(pl.cap, rows_cap(q.numBeads, q.kp, q.rows, kRowsLdsHalf));
    }
    if (!pl.blocks || beads > kRowsMaxBatchBeads || !rows_fits(pl)) return false;
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

hipError_t launch_rows(const RowsPlan &pl, const uint32_t *hash, uint32_t *wormRows, const float4 *pos, float4 *force,
                       uint32_t *ids, uint32_t *off, uint32_t *sCell, float4 *sPos, uint32_t N, const KP &kp,
                       hipStream_t st) {
    const RowsArgs a{hash, wormRows, pos, force, ids, off, sCell, sPos};
    const hipError_t e = grant_lds(reinterpret_cast<const void *>(&k_rows), pl.lds);
    if (e != hipSuccess) return e;
    NW_LAUNCH(k_rows, dim3(pl.blocks), dim3(kRowsBlock), pl.lds, st, a, N, pl.rows, pl.cap, pl.cells, kp);
    return hipGetLastError();
}

}  // namespace nw
