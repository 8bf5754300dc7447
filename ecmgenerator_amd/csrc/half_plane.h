// half_plane.h -- the ORCA half-plane of one agent against another, in the
// branching form that covers every operand and in a branch-free form for the
// common ones (device code).
#pragma once

#include "ecm_geom.h"
#include "sim_device.h"

namespace ecm {

// Agent half-plane (ORCA.cpp:339-423)
__device__ void agent_constraint(const DevState& s, V2 position, V2 velocity, float rad,
                                 float4 q, float2 qv, V2& outP, V2& outN) {
    const float T = s.time_horizon;
    const float combined = q.z + rad;
    V2 VOPos;
    float VORadius;
    if (s.inv_time_horizon != 0.0f) {           // T a power of two: the same values without dividing
        const float iT = s.inv_time_horizon;
        VOPos = mk((q.x - position.x) * iT, (q.y - position.y) * iT);
        VORadius = combined * iT;
    } else {
        VOPos = mk((q.x - position.x) / T, (q.y - position.y) / T);
        VORadius = combined / T;
    }
    float VOPosLength = len(VOPos);
    V2 relVel = mk(velocity.x - qv.x, velocity.y - qv.y);
    V2 relPos = mk(q.x - position.x, q.y - position.y);
    float relPosLength = len(relPos);
    if (relPosLength < combined) {
        const V2 w = relVel - relPos / s.dt;
        const float wl = len(w);
        const V2 uw = w / wl;
        const V2 U = uw * (combined / s.dt - wl);
        outP = velocity + U * 0.5f; outN = uw;
        return;
    }
    float half = atan_f(VORadius / VOPosLength);
    V2 VOLeftLeg, VORightLeg;
    rotate_pm(VOPos, half, VOLeftLeg, VORightLeg);     // rotate(VOPos, +-half)
    float sqFromCentre = sq_dist(VOPos, relVel);
    bool below = det(VOLeftLeg - VOPos, relVel - VOPos) > 0;
    if (below) {
        float distToEdge = VORadius - sqrtf(sqFromCentre);
        V2 ln = normalize(relVel - VOPos);
        outP = velocity + (ln * distToEdge) * 0.5f; outN = ln;
    } else {
        const V2 lperp = left(VOPos) / VOPosLength;
        if (dot(lperp, relVel) >= 0) {
            const V2 ll = normalized(VOLeftLeg);
            const V2 U = ll * dot(relVel, ll) - relVel;
            outP = velocity + U * 0.5f; outN = left(ll);
        } else {
            const V2 rl = normalized(VORightLeg);
            const V2 U = rl * dot(relVel, rl) - relVel;
            outP = velocity + U * 0.5f; outN = right(rl);
        }
    }
}

// agent_constraint without a branch, for the common operands: false where one
// of them is outside the ranges of the cheap quotients (tiny, huge or NaN
// coordinates, the side of a leg within rounding), and the caller takes
// agent_constraint then.  Needs s.inv_dt.  The three kinds (colliding, on the
// cutoff disc, on a leg) each normalise one vector: it is selected first and
// normalised once.  With T a power of two the scaled length is the length
// scaled, so one root serves both, and the legs' angle is that of the
// unscaled radius and distance.  About 170 instructions against 330 in a
// wavefront whose lanes meet every kind.
__device__ __forceinline__ bool agent_constraint_common(const DevState& s, V2 position, V2 velocity, float rad,
                                                        float4 q, float2 qv, V2& outP, V2& outN) {
    const float combined = q.z + rad;
    const V2 relVel = mk(velocity.x - qv.x, velocity.y - qv.y);
    const V2 relPos = mk(q.x - position.x, q.y - position.y);
    const float S = len2(relPos);
    const float y = __builtin_amdgcn_rsqf(S);
    const float l = root_from(S, y);
    const bool colliding = l < combined;
    const V2 VOPos = relPos * s.inv_time_horizon;
    V2 left_leg, right_leg;
    rotate_pm(VOPos, atan_unit(quot(combined, l, recip_from(l, y))), left_leg, right_leg);
    const V2 w = relVel - VOPos;
    const bool below = det(left_leg - VOPos, w) > 0;
    // sign of dot(left(VOPos) / |VOPos|, relVel): that of the undivided
    // product, unless it is within the rounding of the divided one
    const float c0 = VOPos.y * relVel.x, c1 = VOPos.x * relVel.y, side = c1 - c0;
    const bool sure = fabsf(side) > __builtin_fmaf(0x1p-20f, fabsf(c0) + fabsf(c1), 0x1p-60f);
    const bool on_left = side > 0.0f, disc = colliding || below;
    const V2 wc = relVel - quot(relPos, s.dt, s.inv_dt);
    const V2 leg = mk(on_left ? left_leg.x : right_leg.x, on_left ? left_leg.y : right_leg.y);
    const V2 v = mk(colliding ? wc.x : (below ? w.x : leg.x), colliding ? wc.y : (below ? w.y : leg.y));
    const float R = colliding ? quot(combined, s.dt, s.inv_dt) : combined * s.inv_time_horizon;
    const float Sv = len2(v);
    const float yv = __builtin_amdgcn_rsqf(Sv);
    const float lv = root_from(Sv, yv);
    const V2 u = quot(v, lv, recip_from(lv, yv));
    const float f = disc ? R - lv : dot(relVel, u);
    V2 U = u * f;
    U = mk(disc ? U.x : U.x - relVel.x, disc ? U.y : U.y - relVel.y);
    outP = velocity + U * 0.5f;
    outN = mk(disc ? u.x : (on_left ? -u.y : u.y), disc ? u.y : (on_left ? u.x : -u.x));
    return exp_within(S, -60, 60) & exp_within(combined, -60, 60) & not_tiny(relPos) & !all_ones(l) &
           exp_within(Sv, -60, 60) & not_tiny(v) & !all_ones(lv) & (disc | sure);
}

}  // namespace ecm
