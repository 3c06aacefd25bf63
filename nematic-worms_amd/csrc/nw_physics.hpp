// nw_physics.hpp -- device physics shared by the per-call kernels
// (nw_kernels.hip) and the fused step kernels (nw_fused.hip): boundaries,
// the WCA magnitude, stencil folding, cross-lane shuffles, per-element uniforms.
#pragma once

#include "nw_device.hpp"

namespace nw {

// ---------------------------------------------------------------------------
// boundaries (particles_kernel_impl.cuh:34-68)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void periodic_bc(float &r, float L0, float L) {
    if (r < L0) r += L;
    else if (r > L + L0) r -= L;
}

__device__ __forceinline__ void damped_wall(float &r, float &v, float coef, float L0, float L, float R) {
    if (r < L0 + R) {
        r = L0 + R;
        v *= coef;
    } else if (r > (L + L0) - R) {
        r = (L + L0) - R;
        v *= coef;
    }
}

// noslipWallBoundary: undo the whole step displacement, pin the axis at the
// wall and keep only the reflected normal velocity component.
__device__ __forceinline__ void noslip_wall(f3 &pos, int axis, f3 &vel, f3 dr, f3 N, float L0, float L, float R) {
    float r = axis == 0 ? pos.x : pos.y;
    bool hit = false;
    float target = 0.0f;
    if (r < L0 + R) {
        hit = true;
        target = L0 + R;
    } else if (r > (L + L0) - R) {
        hit = true;
        target = (L + L0) - R;
    }
    if (hit) {
        pos -= dr;
        if (axis == 0) pos.x = target; else pos.y = target;
        vel = mk(-vel.x * N.x, -vel.y * N.y, -vel.z * N.z);
    }
}

// periodic_bc without a branch
__device__ __forceinline__ float periodic_select(float r, float L0, float L) {
    return r < L0 ? r + L : (r > L + L0 ? r - L : r);
}

__device__ __forceinline__ void apply_boundaries(const SimParams &p, f3 &pos, f3 &vel, f3 dr, float R) {
    // a box periodic on every axis (PERIODIC is 0): no branch of the lanes
    if ((p.boundaryX | p.boundaryY | p.boundaryZ) == PERIODIC) {
        pos = mk(periodic_select(pos.x, p.origin.x, p.boxSize.x), periodic_select(pos.y, p.origin.y, p.boxSize.y),
                 periodic_select(pos.z, p.origin.z, p.boxSize.z));
        return;
    }
    if (p.boundaryX == PERIODIC) periodic_bc(pos.x, p.origin.x, p.boxSize.x);
    else if (p.boundaryX == WALL) damped_wall(pos.x, vel.x, p.boundaryDamping, p.origin.x, p.boxSize.x, R);
    else if (p.boundaryX == WALL_NO_SLIP)
        noslip_wall(pos, 0, vel, dr, mk(1.f, 0.f, 0.f), p.origin.x, p.boxSize.x, R);

    if (p.boundaryY == PERIODIC) periodic_bc(pos.y, p.origin.y, p.boxSize.y);
    else if (p.boundaryY == WALL) damped_wall(pos.y, vel.y, p.boundaryDamping, p.origin.y, p.boxSize.y, R);
    else if (p.boundaryY == WALL_NO_SLIP)
        noslip_wall(pos, 1, vel, dr, mk(0.f, 1.f, 0.f), p.origin.y, p.boxSize.y, R);

    // the reference has no no-slip branch for z
    if (p.boundaryZ == PERIODIC) periodic_bc(pos.z, p.origin.z, p.boxSize.z);
    else if (p.boundaryZ == WALL) damped_wall(pos.z, vel.z, p.boundaryDamping, p.origin.z, p.boxSize.z, R);
}

// ---------------------------------------------------------------------------
// pair terms and the neighbour stencil (particles_kernel_impl.cuh:427-556)
// ---------------------------------------------------------------------------
struct AxisCells {
    int c[3];
    float w[3];
    int n;
};

// The distinct cells around coordinate g in [0, G) and how often the
// reference's three offsets land on each; the neighbours wrap by selects
__device__ __forceinline__ AxisCells axis_cells_in(int g, uint32_t G, bool onlyCentre) {
    AxisCells a = {{g, g, g}, {0.f, 0.f, 0.f}, 0};  // unused entries: the centre cell, weight 0
    if (onlyCentre) {
        a.c[0] = g;
        a.w[0] = 1.0f;
        a.n = 1;
        return a;
    }
    const int Gi = int(G);
    const int m = g == 0 ? Gi - 1 : g - 1, c = g, p = g + 1 == Gi ? 0 : g + 1;
    if (G >= 3) {
        a.c[0] = m; a.c[1] = c; a.c[2] = p;
        a.w[0] = a.w[1] = a.w[2] = 1.0f;
        a.n = 3;
    } else if (G == 2) {
        a.c[0] = m; a.w[0] = 2.0f;
        a.c[1] = c; a.w[1] = 1.0f;
        a.n = 2;
    } else {
        a.c[0] = c; a.w[0] = 3.0f;
        a.n = 1;
    }
    return a;
}

// 24 eps (2 s^12/r^14 - s^6/r^8) at rr = r^2, with the hardware reciprocal
// (1 ulp): the force is a product of powers of 1/r^2
__device__ __forceinline__ float wca_mag(const NWExtParams &e, float rr) {
    const float inv2 = __builtin_amdgcn_rcpf(rr);
    const float s2 = e.wcaSigma * e.wcaSigma * inv2;
    const float s6 = s2 * s2 * s2;
    return 24.0f * e.wcaEpsilon * inv2 * s6 * (2.0f * s6 - 1.0f);
}

// ---------------------------------------------------------------------------
// cross-lane exchange of chain neighbours
// ---------------------------------------------------------------------------
__device__ __forceinline__ f3 shfl_down3(f3 a, int d) {
    return mk(__shfl_down(a.x, d, 64), __shfl_down(a.y, d, 64), __shfl_down(a.z, d, 64));
}
__device__ __forceinline__ f3 shfl_up3(f3 a, int d) {
    return mk(__shfl_up(a.x, d, 64), __shfl_up(a.y, d, 64), __shfl_up(a.z, d, 64));
}

// The least and the greatest of y (below 2^16) over the lanes of a worm of n
// beads, as (2^16 - 1 - least) << 16 | greatest, in its first lane (pp the
// lane's bead in the worm)
__device__ __forceinline__ uint32_t worm_rows_word(uint32_t y, uint32_t pp, uint32_t n) {
    typedef uint16_t w2 __attribute__((ext_vector_type(2)));
    uint32_t w = (0xffffu - y) << 16 | y;
    for (uint32_t d = 1; d < n; d <<= 1) {
        const uint32_t x = __shfl_down(w, d, 64);
        if (pp + d < n)
            w = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(w2, w), __builtin_bit_cast(w2, x)));
    }
    return w;
}

// x of lane I of this lane's quad
template <int I>
__device__ __forceinline__ float quad_lane(float x) {
    constexpr int ctrl = I | I << 2 | I << 4 | I << 6;  // quad_perm
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xf, 0xf, true));
}
// acc + the four lanes' terms, lane 0's first
__device__ __forceinline__ void add_quad(f3 &acc, f3 t) {
    acc += mk(quad_lane<0>(t.x), quad_lane<0>(t.y), quad_lane<0>(t.z));
    acc += mk(quad_lane<1>(t.x), quad_lane<1>(t.y), quad_lane<1>(t.z));
    acc += mk(quad_lane<2>(t.x), quad_lane<2>(t.y), quad_lane<2>(t.z));
    acc += mk(quad_lane<3>(t.x), quad_lane<3>(t.y), quad_lane<3>(t.z));
}

// ---------------------------------------------------------------------------
// Whole worms packed per 64-lane wavefront: floor(64/n) worms per wave, bead
// p of worm w on lane (w mod wpw) * n + p, the remaining lanes idle.
// ---------------------------------------------------------------------------
struct WaveWorm {
    uint32_t lane, wl, pp, worm, bead;
    bool active;
};

// lanes of wavefront `wave` of a system of W worms of n beads
__device__ __forceinline__ WaveWorm wave_worm_at(uint32_t wave, uint32_t n, uint32_t W) {
    WaveWorm m;
    m.lane = threadIdx.x & 63u;
    const uint32_t wpw = 64u / n;
    m.wl = m.lane / n;
    m.pp = m.lane - m.wl * n;
    m.worm = wave * wpw + m.wl;
    m.active = m.wl < wpw && m.worm < W;
    m.bead = m.worm * n + m.pp;
    return m;
}

__device__ __forceinline__ WaveWorm wave_worm(uint32_t n, uint32_t W) {
    WaveWorm m;
    m.lane = threadIdx.x & 63u;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint32_t wpw = 64u / n;
    m.wl = m.lane / n;
    m.pp = m.lane - m.wl * n;
    m.worm = wave * wpw + m.wl;
    m.active = m.wl < wpw && m.worm < W;
    m.bead = m.worm * n + m.pp;
    return m;
}

// Bonded forces on bead pp (filamentKernel, particles_kernel_impl.cuh:751-818,
// and in chain mode the archived harmonic bonds + drive) added to acc in the
// reference's order: triple pp-2 (its k share), triple pp-1 (j share), triple
// pp (i share), then -bond(pp-1), +bond(pp), +drive.  Lane pp evaluates the
// triple (pp, pp+1, pp+2) and the bond (pp, pp+1) once; the shares of the
// other beads arrive by shuffles.  Every lane of the wave must call this.
// Returns whether the tangent tg is written (the reference writes none for
// n < 3 and no tail tangent for n == 3).
// wantTan = false: the tangent is neither computed nor reported (a caller
// that stores none)
__device__ __forceinline__ bool bonded_lane(const KP &kp, f3 r, uint32_t pp, f3 &acc, f3 &tg, bool wantTan = true) {
    const SimParams &p = kp.p;
    const uint32_t n = p.filamentSize;
    const f3 rn1 = shfl_down3(r, 1);
    // the bond (pp, pp + 1) and its length, once; the bond (pp + 1, pp + 2) is
    // the next lane's, the same values from the same positions.
    // min_image_pair: min_image's value, the wrap tests only when some lane's
    // chain spans half the box
    const f3 r_ij = min_image_pair(p, r, rn1);
    const float dd = dot(r_ij, r_ij), d_ij = sqrtf(dd);
    const f3 r_jk = shfl_down3(r_ij, 1);
    const float dd_jk = __shfl_down(dd, 1, 64), d_jk = __shfl_down(d_ij, 1, 64);

    f3 fi = mk(0.f, 0.f, 0.f), fj = fi, fk = fi;
    const bool hasTriple = n >= 3 && pp + 2u < n;
    if (hasTriple) {
        const float d_ij_jk = dot(r_ij, r_jk);
        const float A = p.bondBendingK / (d_ij * d_jk);
        const f3 B = r_ij * d_ij_jk / dd;
        const f3 C = r_jk * d_ij_jk / dd_jk;
        fi = -A * (r_jk - B);
        fk = -A * (C - r_ij);
        fj = mk(-fi.x - fk.x, -fi.y - fk.y, -fi.z - fk.z);
    }
    const f3 fk_from2 = shfl_up3(fk, 2);
    const f3 fj_from1 = shfl_up3(fj, 1);

    const bool chain = kp.e.bondedMode == NW_BONDED_CHAIN;
    f3 fb = mk(0.f, 0.f, 0.f), drive = fb;
    if (chain && pp + 1u < n) {
        fb = (p.bondSpringK * (d_ij - p.bondSpringL) / d_ij) * r_ij;
        drive = (kp.e.driveForce / d_ij) * r_ij;
    }
    const f3 fb_prev = shfl_up3(fb, 1);

    if (pp >= 2u) acc += fk_from2;
    if (pp >= 1u) acc += fj_from1;
    if (hasTriple) acc += fi;
    if (chain) {
        if (pp >= 1u) acc -= fb_prev;
        if (pp + 1u < n) {
            acc += fb;
            acc += drive;
        }
    }
    if (n < 3 || !wantTan) return false;
    const f3 rp1 = shfl_up3(r, 1);
    if (pp == 0u) tg = tangent_of(p, r, rn1);
    else if (pp + 1u < n) tg = tangent_of(p, rp1, rn1);
    else {
        tg = tangent_of(p, rp1, r);
        return n > 3u;
    }
    return true;
}

// element e of a uniform draw at `offset` (lane e%4 of block offset + e/4)
__device__ __forceinline__ float uniform_at(uint64_t seed, uint64_t offset, uint32_t e) {
    const u4 b = philox_block(seed, offset + (e >> 2));
    const uint32_t k = e & 3u;
    const uint32_t x = k == 0 ? b.x : k == 1 ? b.y : k == 2 ? b.z : b.w;
    return u01(x);
}

}  // namespace nw
