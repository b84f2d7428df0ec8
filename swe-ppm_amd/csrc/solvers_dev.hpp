// solvers_dev.hpp -- per-edge Riemann solvers as CDNA4 device code.
//
// Interface of the reference's solver call sites
//   solver.computeNetUpdates(hL, hR, huL, huR, bL, bR,
//                            hNetL, hNetR, huNetL, huNetR, maxEdgeSpeed)
// (src/blocks/SWE_DimensionalSplittingMpi.cpp:403-410), whose bodies live in
// the un-vendored TUM-I5/swe_solvers submodule.  The arithmetic here is this
// library's own statement of the published methods:
//   f-wave   -- Bale, LeVeque, Mitran, Rossmanith 2002, Einfeldt speeds;
//   AugRie   -- George 2008 (J. Comput. Phys. 227), three f-waves with the
//               steady-state wave removed, wet/dry walls and inundation,
//               Newton middle state for shock cases;
//   HLLE     -- Einfeldt 1988 in fluctuation form;
//   Hybrid   -- f-wave when both depths >= kHybridTol, AugRie otherwise.
//
// Written for wave64 execution: the wet/dry and wave-direction decisions are
// predicates folded into selects; only the expensive, spatially clustered
// paths (wet/dry wall test, Newton loops) are real branches, which stay
// uniform inside most waves.  Every floating-point expression keeps one fixed
// evaluation order (no contraction in parity builds), so that results are
// reproducible against an IEEE CPU evaluation of the same formulas.
#pragma once

#include <hip/hip_runtime.h>

#include "exact_math.hpp"
#include "swe_common.h"

namespace swe {
namespace dev {

// std::min / std::max semantics (first operand wins ties), not fminf/fmaxf.
__device__ __forceinline__ float smin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float smax(float a, float b) { return (a < b) ? b : a; }

struct EdgeOut {
    float hL, hR, huL, huR, speed;
};

// One side of an edge: depth, normal momentum, bathymetry and the per-cell
// quantities every edge touching the cell needs.  They are computed once per
// cell (cell_side) and reused by its four edges; the values are the same
// IEEE results each edge would compute itself.
struct Side {
    float h, hu, b;
    float u;    // hu (1/h) (normal velocity; meaningless for dry cells)
    float c;    // sqrt(g h)
    float sq;   // sqrt(h)
    float inv;  // 1 / h (the augmented solver's middle state divides by both depths)
};

template <class A = Ieee>
__device__ __forceinline__ Side cell_side(float h, float hu, float b) {
    Side s;
    s.h = h;
    s.hu = hu;
    s.b = b;
    s.inv = A::rcp(h);
    s.u = hu * s.inv;
    s.sq = A::sqrt(h);
    s.c = kSqrtGravity * s.sq;
    return s;
}

// Add one f-wave to the side its speed points to; a wave of (near) zero speed
// is shared equally.  Expressed as selects of the three branch results.
__device__ __forceinline__ void acc_wave(float s, float zh, float zhu, EdgeOut& o) {
    const bool left = s < -kZeroTol;
    const bool right = s > kZeroTol;
    const float hzh = 0.5f * zh;
    const float hzhu = 0.5f * zhu;
    const float hL = left ? o.hL + zh : (right ? o.hL : o.hL + hzh);
    const float huL = left ? o.huL + zhu : (right ? o.huL : o.huL + hzhu);
    const float hR = right ? o.hR + zh : (left ? o.hR : o.hR + hzh);
    const float huR = right ? o.huR + zhu : (left ? o.huR : o.huR + hzhu);
    o.hL = hL;
    o.huL = huL;
    o.hR = hR;
    o.huR = huR;
}

// A dry neighbour of an f-wave / HLLE edge is a reflecting wall: the wet
// state mirrored (h, -hu, b; the velocity negates exactly).
struct Mirrored {
    Side L, R;
    bool dryL, dryR, mirrorR;
};
__device__ __forceinline__ Mirrored mirror_dry(const Side& L, const Side& R) {
    Mirrored m;
    m.dryL = L.h < kDryTol;
    m.dryR = R.h < kDryTol;
    m.mirrorR = !m.dryL && m.dryR;
    m.L.h = m.dryL ? R.h : L.h;
    m.L.hu = m.dryL ? -R.hu : L.hu;
    m.L.b = m.dryL ? R.b : L.b;
    m.L.u = m.dryL ? -R.u : L.u;
    m.L.c = m.dryL ? R.c : L.c;
    m.L.sq = m.dryL ? R.sq : L.sq;
    m.L.inv = m.dryL ? R.inv : L.inv;
    m.R.h = m.mirrorR ? L.h : R.h;
    m.R.hu = m.mirrorR ? -L.hu : R.hu;
    m.R.b = m.mirrorR ? L.b : R.b;
    m.R.u = m.mirrorR ? -L.u : R.u;
    m.R.c = m.mirrorR ? L.c : R.c;
    m.R.sq = m.mirrorR ? L.sq : R.sq;
    m.R.inv = m.mirrorR ? L.inv : R.inv;
    return m;
}

// ---------------------------------------------------------------------------
// f-wave
// ---------------------------------------------------------------------------
template <class A = Ieee>
__device__ __forceinline__ EdgeOut fwave(const Side& Lin, const Side& Rin) {
    const Mirrored m = mirror_dry(Lin, Rin);
    const Side& L = m.L;
    const Side& R = m.R;
    const float hRoe = 0.5f * (L.h + R.h);
    const float uRoe = A::div(L.u * L.sq + R.u * R.sq, L.sq + R.sq);
    const float cRoe = A::sqrt(kGravity * hRoe);
    const float s1 = smin(L.u - L.c, uRoe - cRoe);
    const float s2 = smax(R.u + R.c, uRoe + cRoe);

    const float df1 = R.hu - L.hu;
    const float fR = R.hu * R.u + 0.5f * kGravity * R.h * R.h;
    const float fL = L.hu * L.u + 0.5f * kGravity * L.h * L.h;
    const float df2 = (fR - fL) + 0.5f * kGravity * (L.h + R.h) * (R.b - L.b);
    const float invDs = A::rcp(s2 - s1);
    const float beta1 = (s2 * df1 - df2) * invDs;
    const float beta2 = (df2 - s1 * df1) * invDs;

    EdgeOut o{0.f, 0.f, 0.f, 0.f, 0.f};
    acc_wave(s1, beta1, beta1 * s1, o);
    acc_wave(s2, beta2, beta2 * s2, o);
    o.hL = m.dryL ? 0.f : o.hL;
    o.huL = m.dryL ? 0.f : o.huL;
    o.hR = m.mirrorR ? 0.f : o.hR;
    o.huR = m.mirrorR ? 0.f : o.huR;
    o.speed = smax(fabsf(s1), fabsf(s2));
    if (m.dryL && m.dryR) o = EdgeOut{0.f, 0.f, 0.f, 0.f, 0.f};
    return o;
}

// ---------------------------------------------------------------------------
// Middle state of the Riemann problem: phi(h) = du + f(h; hMin) + f(h; hMax)
// with shock curves (h-k) sqrt(g/2 (1/h + 1/k)) and rarefaction curves
// 2 (sqrt(g h) - sqrt(g k)).  Two rarefactions: closed form.  Otherwise one
// branch-free Newton loop serves both the two-shock case (from hMax) and the
// shock+rarefaction case (from hMin): the curve towards hMax is selected per
// lane, and its two square roots share one instruction slot.  The
// derivative's two quotients share one division, num / den, and the step
// phi / dphi is taken with both sides scaled by den, so an iteration divides
// twice (1/h and the step).  phi is increasing and
// concave on the search interval, so the iterates increase monotonically.
// cL, cR are the cells' celerities sqrt(g) sqrt(h); invL, invR are 1 / hL,
// 1 / hR, computed once per cell.
// ReuseFirst: the first iteration starts at hMax or hMin, where 1/h is known
// and, for two shocks, one of the two curve square roots (the bracket's own
// quantities); with ReuseFirst it takes them instead of recomputing them, so
// it costs no division and one square root (two shocks) or two (shock and
// rarefaction).  The values are the ones the loop computes, so both forms give
// identical results (the single-block sweeps and the batched kernels use it).
// The curves of the next iterate are evaluated at the end of the loop's body,
// so that it exists once in the code.
// ---------------------------------------------------------------------------
struct Middle {
    float hm, s1m, s2m;
};

template <bool ReuseFirst = false, class A = Ieee>
__device__ __forceinline__ Middle middle_state(float hL, float hR, float uL, float uR, float cL, float cR, float invL,
                                               float invR) {
    const float hMin = smin(hL, hR);
    const float hMax = smax(hL, hR);
    const float du = uR - uL;
    Middle m;
    if (hMin < kDryTol) {
        m.hm = 0.f;
        m.s1m = uR + uL - 2.f * cR + 2.f * cL;
        m.s2m = m.s1m;
        return m;
    }
    const float cMin = (hR < hL) ? cR : cL;
    const float cMax = (hL < hR) ? cR : cL;
    const float invMin = (hR < hL) ? invR : invL;  // 1 / hMin
    const float invMax = (hL < hR) ? invR : invL;  // 1 / hMax
    const float halfG = 0.5f * kGravity;
    const float quarterG = 0.25f * kGravity;
    const float fMin = du + 2.f * (cMin - cMax);
    const float gMaxMin = A::sqrt(halfG * (invMax + invMin));
    const float fMax = du + (hMax - hMin) * gMaxMin;
    if (fMin > 0.f) {
        const float a = smax(0.f, -du + 2.f * (cL + cR));
        m.hm = A::div(a * a, 16.f * kGravity);
        const float cm = A::sqrt0(kGravity * m.hm);
        m.s1m = uL + 2.f * cL - 3.f * cm;
        m.s2m = uR - 2.f * cR + 3.f * cm;
        return m;
    }
    const bool shocks = fMax <= 0.f;
    float h = shocks ? hMax : hMin;
    float invH = 0.f, gMin = 0.f, s2 = 0.f;
    if constexpr (ReuseFirst) {
        // at h = hMax the shock curve of hMin is gMaxMin and the new root is
        // gMax(hMax); at h = hMin the new root is gMin(hMin) and the
        // rarefaction root sqrt(g hMin) is taken as the loop takes it (the
        // cell's celerity cMin = sqrt(g) sqrt(hMin) can differ in the last bit)
        invH = shocks ? invMax : invMin;
        const float r0 = A::sqrt(halfG * (invH + invH));
        gMin = shocks ? gMaxMin : r0;
        s2 = shocks ? r0 : A::sqrt(kGravity * hMin);
    }
    auto curves = [&] {
        invH = A::rcp(h);
        gMin = A::sqrt(halfG * (invH + invMin));
        // shocks: gMax(h); shock+rarefaction: sqrt(g h)
        s2 = A::sqrt(shocks ? halfG * (invH + invMax) : kGravity * h);
    };
    if constexpr (!ReuseFirst) curves();
#pragma unroll 1
    for (int it = 1;; ++it) {
        const float t2 = shocks ? (h - hMax) * s2 : 2.f * (s2 - cMax);
        const float phi = (du + (h - hMin) * gMin) + t2;
        const float q = shocks ? s2 : 1.f;
        const float num = (h - hMin) * q + (shocks ? (h - hMax) * gMin : 0.f);
        const float den = gMin * q;
        const float first = gMin + (shocks ? s2 : s2 * invH);
        // phi / (first - quarterG invH^2 num / den) with both terms scaled by
        // den: one division instead of two
        const float step = A::div(phi * den, first * den - quarterG * invH * invH * num);
        h = h - step;
        if (fabsf(step) <= kNewtonTol * h || it == kMaxNewton) break;
        curves();
    }
    m.hm = h;
    const float cm = A::sqrt(kGravity * h);
    if (shocks) {
        const bool leftIsMin = !(hR < hL);
        const float gL = leftIsMin ? gMin : s2;
        const float gR = leftIsMin ? s2 : gMin;
        const float u1m = uL - (h - hL) * gL;
        const float u2m = uR + (h - hR) * gR;
        m.s1m = u1m - cm;
        m.s2m = u2m + cm;
    } else if (hL > hR) {
        m.s1m = uL + 2.f * cL - 3.f * cm;
        m.s2m = uL + 2.f * cL - cm;
    } else {
        m.s1m = uR - 2.f * cR + cm;
        m.s2m = uR - 2.f * cR + 3.f * cm;
    }
    return m;
}

// ---------------------------------------------------------------------------
// Augmented Riemann solver.  MiddleFn computes (hm, s1m, s2m) for the main
// Riemann problem of a wet-wet or inundation edge; the exact Newton
// middle_state is the default, the learned surrogate plugs in here.
// ---------------------------------------------------------------------------
template <bool ReuseFirst, class A = Ieee>
struct ExactMiddle {
    using Math = A;
    static constexpr bool kDefers = false;
    __device__ __forceinline__ Middle operator()(float hL, float hR, float uL, float uR, float cL, float cR,
                                                 float invL, float invR, float, float) const {
        return middle_state<ReuseFirst, A>(hL, hR, uL, uR, cL, cR, invL, invR);
    }
};

// Wet/dry handling of the augmented solver (George 2008): a dry side next to
// a wet one is either a wall (the wet side's middle state cannot reach its
// bed: reflect) or inundated (the bed step is cut to the water surface).
struct AugPrep {
    float hL, huL, uL, cL, bL, invL;
    float hR, huR, uR, cR, bR, invR;
    bool wallL, wallR, dryBoth;
};

template <class A = Ieee>
__device__ __forceinline__ AugPrep augrie_prepare(const Side& Lin, const Side& Rin) {
    const bool dryLin = Lin.h < kDryTol;
    const bool dryRin = Rin.h < kDryTol;
    AugPrep p;
    p.dryBoth = dryLin && dryRin;
    p.hL = dryLin ? 0.f : Lin.h;
    p.huL = dryLin ? 0.f : Lin.hu;
    p.uL = dryLin ? 0.f : Lin.u;
    p.cL = dryLin ? 0.f : Lin.c;
    p.bL = Lin.b;
    p.invL = Lin.inv;  // a dry side never reaches the divisions
    p.hR = dryRin ? 0.f : Rin.h;
    p.huR = dryRin ? 0.f : Rin.hu;
    p.uR = dryRin ? 0.f : Rin.u;
    p.cR = dryRin ? 0.f : Rin.c;
    p.bR = Rin.b;
    p.invR = Rin.inv;
    p.wallL = false;
    p.wallR = false;
    if ((dryLin || dryRin) && !p.dryBoth) {
        if (dryRin) {
            const Middle t = middle_state<false, A>(p.hL, p.hL, p.uL, -p.uL, p.cL, p.cL, p.invL, p.invL);
            const float hTest = smax(p.hL, t.hm);
            if (hTest + p.bL < p.bR) {
                p.wallR = true;
                p.hR = p.hL;
                p.huR = -p.huL;
                p.uR = -p.uL;
                p.cR = p.cL;
                p.invR = p.invL;
                p.bR = p.bL;
            } else if (p.hL + p.bL < p.bR) {
                p.bR = p.hL + p.bL;
            }
        } else {
            const Middle t = middle_state<false, A>(p.hR, p.hR, -p.uR, p.uR, p.cR, p.cR, p.invR, p.invR);
            const float hTest = smax(p.hR, t.hm);
            if (hTest + p.bR < p.bL) {
                p.wallL = true;
                p.hL = p.hR;
                p.huL = -p.huR;
                p.uL = -p.uR;
                p.cL = p.cR;
                p.invL = p.invR;
                p.bL = p.bR;
            } else if (p.hR + p.bR < p.bL) {
                p.bL = p.hR + p.bR;
            }
        }
    }
    return p;
}

// A still edge: both cells hold at least kStillTol of water, zero normal
// momentum on both sides, the same free surface h + b in single precision,
// and depths within a factor kStillRatio.  It is a lake at rest, whose exact
// Riemann solution carries no flux: the solver returns zero net updates and
// the speed the full decomposition reports, max(|sE1|, |sE2|) with
// sE1 = min(-cL, -cHat), sE2 = max(cR, cHat) (at rest u = uHat = 0, and for
// depths within a factor 2 the middle-state speeds never replace the
// Einfeldt speeds: s2m > 0 > sE1 and s1m < 0 < sE2).  Still water thus stays
// exactly still, and a wave whose edges are all still skips the middle state
// and the decomposition.  In a wave that mixes still and moving edges every
// lane runs the decomposition and the still lanes take the still result at
// the end: the learned middle state runs its network for the whole wave
// and must be reached with every lane active.
__device__ __forceinline__ bool still_edge(const Side& L, const Side& R) {
    return L.h >= kStillTol && R.h >= kStillTol && L.hu == 0.f && R.hu == 0.f && L.h + L.b == R.h + R.b &&
           L.h <= kStillRatio * R.h && R.h <= kStillRatio * L.h;
}

template <class A = Ieee>
__device__ __forceinline__ float still_speed(const Side& L, const Side& R) {
    const float cHat = A::sqrt(kGravity * 0.5f * (R.h + L.h));
    const float sE1 = smin(-L.c, -cHat);
    const float sE2 = smax(R.c, cHat);
    return smax(fabsf(sE1), fabsf(sE2));
}

template <typename MiddleFn>
__device__ __forceinline__ EdgeOut augrie_with(const Side& Lin, const Side& Rin, const MiddleFn& middle) {
    using A = typename MiddleFn::Math;
    const bool still = still_edge(Lin, Rin);
    if (__all(still)) return EdgeOut{0.f, 0.f, 0.f, 0.f, still_speed<A>(Lin, Rin)};
    const AugPrep p = augrie_prepare<A>(Lin, Rin);
    const bool dryBoth = p.dryBoth;
    const bool wallL = p.wallL, wallR = p.wallR;
    const float hL = p.hL, huL = p.huL, uL = p.uL, cL = p.cL, bL = p.bL;
    const float hR = p.hR, huR = p.huR, uR = p.uR, cR = p.cR, bR = p.bR;

    const float uHat = A::div(cL * uL + cR * uR, cL + cR);
    const float cHat = A::sqrt(kGravity * 0.5f * (hR + hL));
    const float sE1 = smin(uL - cL, uHat - cHat);
    const float sE2 = smax(uR + cR, uHat + cHat);

    const Middle mid = middle(hL, hR, uL, uR, cL, cR, p.invL, p.invR, bL, bR);

    const float l1 = smin(sE1, mid.s2m);
    const float l3 = smax(sE2, mid.s1m);
    const float l2 = 0.5f * (l1 + l3);
    const float dl = l3 - l1;
    const float invDl = A::rcp(dl);
    const float hStarHLL = smax((huL - huR + l3 * hR - l1 * hL) * invDl, 0.f);

    const float dh = hR - hL;
    const float dhu = huR - huL;
    const float phiL = huL * uL + 0.5f * kGravity * hL * hL;
    const float phiR = huR * uR + 0.5f * kGravity * hR * hR;
    const float dphi = phiR - phiL;
    const float db = bR - bL;

    const float hBar = smax(0.5f * (hL + hR), 0.f);
    const float uSum = uL + uR;
    const float s1s2bar = 0.25f * uSum * uSum - kGravity * hBar;
    const float s1s2tilde = smax(0.f, uL * uR) - kGravity * hBar;
    const float ct = kCriticalTol;

    const bool sonic = (fabsf(s1s2bar) <= ct) || (s1s2bar * s1s2tilde <= ct) || (s1s2bar * l1 * l3 <= ct) ||
                       (smin(fabsf(l1), fabsf(l3)) < ct) || ((l1 < 0.f) && (mid.s1m > 0.f)) ||
                       ((l3 > 0.f) && (mid.s2m < 0.f)) || ((uL + cL) * (uR + cR) < 0.f) ||
                       ((uL - cL) * (uR - cR) < 0.f);

    const float invBar = A::rcp(s1s2bar);
    float ddh = sonic ? -db : db * kGravity * hBar * invBar;
    const bool caseA = (l1 < -ct) && (l3 > ct);
    const bool caseB = !caseA && (l1 >= ct);
    const bool caseC = !caseA && !caseB && (l3 <= -ct);
    if (caseA || caseB || caseC) {
        const float hsd = hStarHLL * dl;
        const float inv13 = A::rcp(l1 * l3);
        const float dA = hsd * l1 * inv13;  // hStarHLL dl / l3
        const float dB = hsd * l3 * inv13;  // hStarHLL dl / l1
        const float hiBound = caseA ? dA : (caseB ? dB : hR);
        const float loBound = caseA ? dB : (caseB ? -hL : dA);
        ddh = smin(ddh, hiBound);
        ddh = smax(ddh, loBound);
    }

    float ddphi = sonic ? -kGravity * hBar * db : -db * kGravity * hBar * s1s2tilde * invBar;
    const float pL = -hL * db;
    const float pR = -hR * db;
    ddphi = smin(ddphi, kGravity * smax(pL, pR));
    ddphi = smax(ddphi, kGravity * smin(pL, pR));

    const float del1 = dh - ddh;
    const float del2 = dhu;
    const float del3 = dphi - ddphi;

    const float l1sq = l1 * l1;
    const float l3sq = l3 * l3;
    const float beta1 = (l3 * del1 - del2) * invDl;
    const float beta3 = (del2 - l1 * del1) * invDl;
    const float beta2 = del3 - (beta1 * l1sq + beta3 * l3sq);

    const bool kill1 = wallL;
    const bool kill2 = wallL || wallR;
    const bool kill3 = wallR;
    const float z1h = kill1 ? 0.f : beta1 * l1;
    const float z1hu = kill1 ? 0.f : beta1 * l1sq;
    const float s1 = kill1 ? 0.f : l1;
    const float z2hu = kill2 ? 0.f : beta2;
    const float s2 = kill2 ? 0.f : l2;
    const float z3h = kill3 ? 0.f : beta3 * l3;
    const float z3hu = kill3 ? 0.f : beta3 * l3sq;
    const float s3 = kill3 ? 0.f : l3;

    EdgeOut o{0.f, 0.f, 0.f, 0.f, 0.f};
    acc_wave(s1, z1h, z1hu, o);
    acc_wave(s2, 0.f, z2hu, o);
    acc_wave(s3, z3h, z3hu, o);
    o.speed = smax(fabsf(s1), fabsf(s3));
    if (dryBoth) o = EdgeOut{0.f, 0.f, 0.f, 0.f, 0.f};
    // a middle function that defers the edge returns a negative depth: the
    // edge is marked by a negative speed and solved again elsewhere
    if constexpr (MiddleFn::kDefers)
        if (mid.hm < 0.f) o.speed = -1.f;
    if (still) o = EdgeOut{0.f, 0.f, 0.f, 0.f, still_speed<A>(Lin, Rin)};
    return o;
}

template <bool ReuseFirst = false, class A = Ieee>
__device__ __forceinline__ EdgeOut augrie(const Side& L, const Side& R) {
    return augrie_with(L, R, ExactMiddle<ReuseFirst, A>());
}

// ---------------------------------------------------------------------------
// HLLE in fluctuation form, surface-gradient diffusion (well-balanced)
// ---------------------------------------------------------------------------
template <class A = Ieee>
__device__ __forceinline__ EdgeOut hlle(const Side& Lin, const Side& Rin) {
    const Mirrored m = mirror_dry(Lin, Rin);
    const Side& L = m.L;
    const Side& R = m.R;
    const float uRoe = A::div(L.u * L.sq + R.u * R.sq, L.sq + R.sq);
    const float cRoe = A::sqrt(kGravity * 0.5f * (L.h + R.h));
    const float sL = smin(smin(L.u - L.c, uRoe - cRoe), 0.f);
    const float sR = smax(smax(R.u + R.c, uRoe + cRoe), 0.f);
    const float df1 = R.hu - L.hu;
    const float fR = R.hu * R.u + 0.5f * kGravity * R.h * R.h;
    const float fL = L.hu * L.u + 0.5f * kGravity * L.h * L.h;
    const float df2 = (fR - fL) + 0.5f * kGravity * (L.h + R.h) * (R.b - L.b);
    const float dq1 = (R.h + R.b) - (L.h + L.b);  // surface-gradient form: lake at rest stays at rest
    const float dq2 = R.hu - L.hu;
    const float invDs = A::rcp(sR - sL);
    const float q1 = (sR * dq1 - df1) * invDs;
    const float q2 = (sR * dq2 - df2) * invDs;
    EdgeOut o;
    o.hL = sL * q1;
    o.huL = sL * q2;
    o.hR = df1 - o.hL;
    o.huR = df2 - o.huL;
    o.hL = m.dryL ? 0.f : o.hL;
    o.huL = m.dryL ? 0.f : o.huL;
    o.hR = m.mirrorR ? 0.f : o.hR;
    o.huR = m.mirrorR ? 0.f : o.huR;
    o.speed = smax(fabsf(sL), fabsf(sR));
    if (m.dryL && m.dryR) o = EdgeOut{0.f, 0.f, 0.f, 0.f, 0.f};
    return o;
}

// One edge with solver S.  ReuseFirst selects the form of the Newton loop
// (middle_state), A that of divisions and square roots; the results are the
// same.
template <int S, bool ReuseFirst = false, class A = Ieee>
__device__ __forceinline__ EdgeOut solve_edge(const Side& L, const Side& R) {
    if constexpr (S == SOLVER_FWAVE) return fwave<A>(L, R);
    if constexpr (S == SOLVER_HLLE) return hlle<A>(L, R);
    if constexpr (S == SOLVER_HYBRID)
        if (L.h >= kHybridTol && R.h >= kHybridTol) return fwave<A>(L, R);
    if constexpr (S == SOLVER_AUGRIE || S == SOLVER_HYBRID) return augrie<ReuseFirst, A>(L, R);
}

// Solver with per-kernel state, built once at kernel start from an optional
// parameter block (the learned middle state keeps its network weights in
// registers; the exact solvers have no state).  kNormalForm: the sweeps solve
// the edges of ordinary cells with NormalRange (column_edges in kernels_u.hpp).
template <int S, bool ReuseFirst = false>
struct SolverCtx {
    static constexpr bool kNormalForm = true;
    __device__ __forceinline__ explicit SolverCtx(const unsigned*) {}
    template <class A = Ieee>
    __device__ __forceinline__ EdgeOut solve(const Side& L, const Side& R) const {
        return solve_edge<S, ReuseFirst, A>(L, R);
    }
};

// Cells whose edges may be solved with NormalRange: depth and bed below 2^40 and,
// on a wet cell, velocities below 2^20 in sum.  A dry cell's momentum, velocity,
// celerity and 1/h reach no result (the augmented solver sets them to zero, the
// others mirror the wet side, and an edge between two dry cells returns zeros),
// so every operand of a wet edge is normal:
//   * h >= 0.01, so celerities lie in [0.3, 2^22] and every sum of two, every
//     depth sum and its root is bounded away from zero;
//   * speeds are below 2^23, and the fastest two of an edge differ by at least
//     2 cHat less their rounding, > 0.3: the divisions by l3 - l1 and s2 - s1;
//   * 1 / (l1 l3) and 1 / s1s2bar are used only where the operands exceed 1e-12;
//   * Newton's depths stay between hMin and about 2^60, its two curve roots
//     above 2^-30, so its denominator lies above 2^-90;
//   * 2 (cL + cR) - du is zero or at least 2^-24, and its square a normal number.
// Numerators below 2^-102 occur in two places, the Roe velocity and the Newton
// step; the first is added to a celerity above 0.2, the second to a depth above
// 0.01, and neither changes the sum in any rounding.  A NaN fails the test.
__device__ __forceinline__ bool in_normal_range(float h, float b, float u, float v) {
    return (fabsf(h) + fabsf(b) <= 0x1p40f) && (h < kDryTol || fabsf(u) + fabsf(v) <= 0x1p20f);
}

// Convenience for raw edge states (one-off evaluations).
template <int S, bool ReuseFirst = false, class A = Ieee>
__device__ __forceinline__ EdgeOut solve_raw(float hL, float hR, float huL, float huR, float bL, float bR) {
    return solve_edge<S, ReuseFirst, A>(cell_side<A>(hL, huL, bL), cell_side<A>(hR, huR, bR));
}

}  // namespace dev
}  // namespace swe
