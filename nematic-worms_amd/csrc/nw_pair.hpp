// nw_pair.hpp -- the pair terms of the excluded-volume pass, shared by its
// kernels (nw_fused.hip: one-layer stencils; nw_pairs.hip: any stencil).
#pragma once

#include "nw_physics.hpp"

namespace nw {

// the bead a thread sums for (its worm and chain index; velocity and tangent
// when the terms read them)
template <int MODE, bool TAN>
struct Owner {
    f3 r, v, t;
    uint32_t fil, ch;
};

// whose a candidate is: the owner itself, of the owner's worm, its chain
// neighbour
struct PairWho {
    bool self, same, bonded;
};
// of the candidate in worm fil2 at place ch2 of its chain
template <int MODE, bool TAN>
__device__ __forceinline__ PairWho pair_who(const Owner<MODE, TAN> &o, uint32_t fil2, uint32_t ch2) {
    const bool same = o.fil == fil2;
    return {same && ch2 == o.ch, same, same && (o.ch + 1u == ch2 || o.ch - 1u == ch2)};
}

// One candidate's terms, MODE 0: the chain bond (bondHookean
// particles_kernel_impl.cuh:466-473) between chain neighbours, else the soft
// sphere (collideParticles :427-462); MODE 1: WCA between different worms;
// TAN: the extensile term (extensileForce :477-487) between different worms.
// The bead itself and, in WCA mode, its own worm are skipped.
// The terms share the separation and its length, and every quotient is of a
// scalar ((-k (L - d)) / d times the separation, not the unit vector's three):
// an exact division is some eleven operations, and the count of roundings
// on the way to a component stays what three divisions made it.
template <int MODE, bool TAN, bool UNIT = false>
__device__ __forceinline__ void add_pair(const KP &kp, const Owner<MODE, TAN> &o, float rc2, float w, f3 &acc,
                                         f3 r2, PairWho who, f3 v2, f3 t2) {
    const SimParams &p = kp.p;
    if (MODE == 0 ? who.self : who.same) return;
    const f3 rel = min_image_pair(p, o.r, r2);
    const float rr = dot(rel, rel);
    f3 t = mk(0.f, 0.f, 0.f);
    if (MODE == 0) {
        const float dist = sqrtf(rr);
        if (who.bonded) {
            t = (-p.bondSpringK * (p.bondSpringL - dist) / dist) * rel;
        } else {
            const float cd = p.particleRadius + p.particleRadius;
            if (dist < cd) {
                const f3 relVel = v2 - o.v;
                const f3 tanVel = relVel - (dot(relVel, rel) / rr) * rel;
                t = (-p.spring * (cd - dist) / dist) * rel;
                t += p.damping * relVel;
                t += p.shear * tanVel;
            }
        }
    } else {
        if (rr < rc2) t = -wca_mag(kp.e, rr) * rel;
    }
    acc += UNIT ? t : w * t;
    if (TAN && !who.same) {
        f3 x = mk(0.f, 0.f, 0.f);
        if (dot(o.t, t2) < -0.5f) x = (-p.activity / (2.0f * sqrtf(rr))) * (o.t - t2);
        acc += UNIT ? x : w * x;
    }
}

// The WCA term of a bead at r of worm fil with the staged record P (position,
// worm in w), evaluated without a branch and masked: a candidate of the bead's
// own worm, at or beyond the cutoff or at a non-finite position gives +0,
// which leaves an accumulator that starts at +0 unchanged (an FP32 sum is -0
// only when both of its terms are)
__device__ __forceinline__ f3 wca_term_masked(const KP &kp, f3 r, uint32_t fil, float rc2, const float4 &P) {
    const f3 rel = min_image_pair(kp.p, r, mk(P));
    const float rr = dot(rel, rel);
    const bool hit = __float_as_uint(P.w) != fil && rr < rc2;
    const f3 f = -wca_mag(kp.e, rr) * rel;
    const uint32_t m = hit ? 0xffffffffu : 0u;
    return mk(__uint_as_float(__float_as_uint(f.x) & m), __uint_as_float(__float_as_uint(f.y) & m),
              __uint_as_float(__float_as_uint(f.z) & m));
}

template <int MODE, bool TAN>
__device__ __forceinline__ Owner<MODE, TAN> load_owner(const KP &kp, uint32_t i, uint32_t me,
                                                       const float4 *__restrict__ sPos,
                                                       const float4 *__restrict__ sVel,
                                                       const float4 *__restrict__ sTan) {
    Owner<MODE, TAN> o;
    o.r = mk(load4(sPos, i));
    o.v = MODE == 0 ? mk(load4(sVel, i)) : mk(0.f, 0.f, 0.f);
    o.t = TAN ? mk(load4(sTan, i)) : mk(0.f, 0.f, 0.f);
    worm_of(kp, me, o.fil, o.ch);
    return o;
}

}  // namespace nw
