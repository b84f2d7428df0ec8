// augrie_normal.hpp -- the augmented solver of solvers_dev.hpp for cells in
// dev::in_normal_range: the same values as dev::augrie, bit for bit, in fewer
// instructions and shorter dependent chains.
//
// What it leaves out or shortens against the general form:
//   * wave-uniform tests skip the still-water test, the dry-cell handling and
//     the wall and supercritical selects where no lane of the wave needs them;
//   * the wall test of a wet cell next to a dry one runs once for both
//     directions (a strip that crosses an island has both in one wave, and the
//     general form runs two Newton loops, one after the other), and uses that
//     the wall problem is symmetric: both curves are one, so an iteration takes
//     one root;
//   * minima and maxima are single instructions (no operand of a live lane is a
//     NaN, and the sign of a zero among them reaches no result), and cMin, cMax,
//     1/hMin and 1/hMax follow from them because correctly rounded roots and
//     reciprocals are monotone;
//   * a product with 2, 4 or 1/4 followed by an addition is one fused
//     operation: the product is exact, so the sum is rounded once either way;
//   * in a wave whose lanes are all subcritical wave 1 goes left and wave 3
//     right, so only wave 2 chooses its side, as a weight of 0, 1/2 or 1.
//   * where both sides are calm (calm_edge) the middle state is not computed.
// On the 2048^2 islands with every cell moving a fused launch issues 83.6 M vector
// instructions in the general form, 61 M with all of the above but the last and
// 35.6 M with it, and takes 156, 103 and 75 us: at the first two bound by vector
// issue, now by half and for the rest by waits for memory.
#pragma once

#include "solvers_dev.hpp"

namespace swe {
namespace dev {

// v_med3_f32 with an infinity: unlike fminf / fmaxf it needs no canonicalised
// operands, which the compiler makes with one more instruction each.  (A known
// infinity would be turned back into fminf / fmaxf.)
__device__ __forceinline__ float scalar_infinity() {
    float x;
    asm("s_mov_b32 %0, 0x7f800000" : "=s"(x));
    return x;
}
__device__ __forceinline__ float vmin(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, -scalar_infinity()); }
__device__ __forceinline__ float vmax(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, scalar_infinity()); }

// Depth of water of depth h (celerity c, inv = 1/h) that runs with velocity un
// into a wall: the middle state of the Riemann problem (h, un | h, -un), as
// middle_state computes it.
__device__ __forceinline__ float wall_depth(float h, float un, float c, float inv) {
    using A = NormalRange;
    const float du = -2.f * un;
    if (du > 0.f) {  // two rarefactions
        const float a = vmax(0.f, __builtin_fmaf(4.f, c, -du));
        return A::div(a * a, 16.f * kGravity);
    }
    float x = h, invX = inv;
    float g = A::sqrt(kGravity * inv);  // sqrt(g/2 (1/x + 1/h)) at x = h
#pragma unroll 1
    for (int it = 1;; ++it) {
        const float t = (x - h) * g;
        const float phi = (du + t) + t;
        const float den = g * g;
        const float step =
            A::div(phi * den, (g + g) * den - 0.25f * kGravity * invX * invX * (t + t));
        x = x - step;
        if (fabsf(step) <= kNewtonTol * x || it == kMaxNewton) return x;
        invX = A::rcp(x);
        g = A::sqrt(0.5f * kGravity * (invX + inv));
    }
}

// True where the middle state is certain to have s1m <= 0 <= s2m, so that it need
// not be computed: with U = max(|uL|, |uR|), cMin and cMax the two celerities,
//   U + 2 cMax < 2.99 cMin   (U < 0.99 cMin and cMax < 1.5 cMin).
// In each of its three forms the middle depth's celerity cm and velocity um bound
// s1m = um - cm from above (s2m = um + cm from below by the mirrored edge):
//   two rarefactions  cm = (2 (cL + cR) - du) / 4, so s1m = uL + 2 cL - 3 cm =
//                     (uL + 3 uR) / 4 + cL / 2 - 3 cR / 2 <= U + cMax / 2 - 3 cMin / 2
//                     (du <= 2 U < 4 cMin: the depth is not cut off at 0);
//   two shocks        cm >= cMax and um <= uL, so s1m <= U - cMax;
//   one of each       cMin <= cm <= cMax.  Left side deep: s1m = uL + 2 cL - 3 cm
//                     <= U + 2 cMax - 3 cMin; right side deep: s1m = uR - 2 cR +
//                     cm <= U - cMax.
// Newton's iterates do not leave these bounds: the depth function is concave and
// increases, so they rise to the root from the start, hMax for two shocks and
// hMin for one of each, whose root lies below hMax.  All operands are normal
// numbers, so rounding moves either side by less than 1e-5 cMin; the test leaves
// 0.01 cMin.  uLm < 0 < uRp follow as well, so min(.., s2m) and max(.., s1m)
// change neither l1 nor l3.  A dry side has c = 0 and fails the test.
__device__ __forceinline__ bool calm_edge(float uL, float uR, float cL, float cR) {
    const float u = vmax(fabsf(uL), fabsf(uR));
    return __builtin_fmaf(2.f, vmax(cL, cR), u) < 2.99f * vmin(cL, cR);
}

// Speeds s1m, s2m of the middle state (middle_state's, whose depth the
// decomposition does not use).
__device__ __forceinline__ void middle_speeds(float hL, float hR, float uL, float uR, float cL, float cR, float invL,
                                              float invR, bool anyDry, float& s1m, float& s2m) {
    using A = NormalRange;
    const float halfG = 0.5f * kGravity;
    const float hMin = vmin(hL, hR);
    const float hMax = vmax(hL, hR);
    const float twoCL = __builtin_fmaf(2.f, cL, uL);   // uL + 2 cL
    const float twoCR = __builtin_fmaf(-2.f, cR, uR);  // uR - 2 cR
    if (anyDry && hMin < kDryTol) {
        s1m = s2m = __builtin_fmaf(2.f, cL, __builtin_fmaf(-2.f, cR, uR + uL));
        return;
    }
    const float du = uR - uL;
    const float cMin = vmin(cL, cR);
    const float cMax = vmax(cL, cR);
    if (__builtin_fmaf(2.f, cMin - cMax, du) > 0.f) {  // two rarefactions
        const float a = vmax(0.f, __builtin_fmaf(2.f, cL + cR, -du));
        const float cm3 = 3.f * A::sqrt0(kGravity * A::div(a * a, 16.f * kGravity));
        s1m = twoCL - cm3;
        s2m = twoCR + cm3;
        return;
    }
    const float invMin = vmax(invL, invR);
    const float invMax = vmin(invL, invR);
    const float gMaxMin = A::sqrt(halfG * (invMax + invMin));
    const bool shocks = du + (hMax - hMin) * gMaxMin <= 0.f;
    float h = shocks ? hMax : hMin;
    float invH = shocks ? invMax : invMin;
    const float r0 = A::sqrt(kGravity * invH);
    float gMin = shocks ? gMaxMin : r0;
    float s2 = shocks ? r0 : A::sqrt(kGravity * hMin);
#pragma unroll 1
    for (int it = 1;; ++it) {
        const float dMin = h - hMin, dMax = h - hMax;
        // (h - hMax) s2 or 2 (s2 - cMax)
        const float t2 = (shocks ? dMax : s2 - cMax) * (shocks ? s2 : 2.f);
        const float phi = (du + dMin * gMin) + t2;
        const float q = shocks ? s2 : 1.f;
        const float num = dMin * q + (shocks ? dMax * gMin : 0.f);
        const float den = gMin * q;
        const float first = gMin + s2 * (shocks ? 1.f : invH);
        const float step = A::div(phi * den, first * den - 0.25f * kGravity * invH * invH * num);
        h = h - step;
        if (fabsf(step) <= kNewtonTol * h || it == kMaxNewton) break;
        invH = A::rcp(h);
        gMin = A::sqrt(halfG * (invH + invMin));
        s2 = A::sqrt(shocks ? halfG * (invH + invMax) : kGravity * h);
    }
    const float cm = A::sqrt(kGravity * h);
    const float cm3 = 3.f * cm;
    const bool leftDeep = hL > hR;
    const float u1m = uL - (h - hL) * (leftDeep ? s2 : gMin);
    const float u2m = uR + (h - hR) * (leftDeep ? gMin : s2);
    const float base = leftDeep ? twoCL : twoCR;
    s1m = (shocks ? u1m : base) - (shocks ? cm : (leftDeep ? cm3 : -cm));
    s2m = (shocks ? u2m : base) + (shocks ? cm : (leftDeep ? -cm : cm3));
}

__device__ __forceinline__ EdgeOut augrie_normal(const Side& L, const Side& R) {
    using A = NormalRange;
    // still edges (still_edge): only where some lane has no normal momentum
    bool still = false;
    const bool anyRest = __any(L.hu == 0.f && R.hu == 0.f);
    if (anyRest) {
        still = still_edge(L, R);
        if (__all(still)) {
            const float cHat = A::sqrt(0.5f * kGravity * (R.h + L.h));
            return EdgeOut{0.f, 0.f, 0.f, 0.f, vmax(vmax(L.c, R.c), cHat)};
        }
    }

    // dry cells (augrie_prepare)
    float hL = L.h, huL = L.hu, uL = L.u, cL = L.c, bL = L.b, invL = L.inv;
    float hR = R.h, huR = R.hu, uR = R.u, cR = R.c, bR = R.b, invR = R.inv;
    const bool dryL = hL < kDryTol, dryR = hR < kDryTol;
    const bool anyDry = __any(dryL || dryR);
    bool wallL = false, wallR = false;
    if (anyDry) {
        hL = dryL ? 0.f : hL;
        huL = dryL ? 0.f : huL;
        uL = dryL ? 0.f : uL;
        cL = dryL ? 0.f : cL;
        hR = dryR ? 0.f : hR;
        huR = dryR ? 0.f : huR;
        uR = dryR ? 0.f : uR;
        cR = dryR ? 0.f : cR;
        if (dryL != dryR) {
            const float hw = dryR ? hL : hR, bw = dryR ? bL : bR, bd = dryR ? bR : bL;
            const float top = wall_depth(hw, dryR ? uL : -uR, dryR ? cL : cR, dryR ? invL : invR);
            const bool wall = vmax(hw, top) + bw < bd;
            const float surface = hw + bw;
            const float cut = !wall && surface < bd ? surface : bd;  // the dry side's bed
            bL = dryL ? cut : bL;
            bR = dryR ? cut : bR;
            wallL = wall && dryL;
            wallR = wall && dryR;
        }
        hL = wallL ? hR : hL;
        huL = wallL ? -huR : huL;
        uL = wallL ? -uR : uL;
        cL = wallL ? cR : cL;
        invL = wallL ? invR : invL;
        bL = wallL ? bR : bL;
        hR = wallR ? hL : hR;
        huR = wallR ? -huL : huR;
        uR = wallR ? -uL : uR;
        cR = wallR ? cL : cR;
        invR = wallR ? invL : invR;
        bR = wallR ? bL : bR;
    }

    const float gh = 0.5f * kGravity * (hR + hL);  // g hBar
    const float cHat = A::sqrt(gh);
    const float uHat = A::div(cL * uL + cR * uR, cL + cR);
    const float uLm = uL - cL, uRp = uR + cR;
    // The middle state enters through the signs of s1m and s2m alone where both
    // sides run well below their celerity and differ little in depth (calm_edge):
    // any values with s1m <= 0 <= s2m leave l1, l3 and the sonic test as they are.
    float s1m = 0.f, s2m = 0.f;
    if (!calm_edge(uL, uR, cL, cR)) middle_speeds(hL, hR, uL, uR, cL, cR, invL, invR, anyDry, s1m, s2m);
    const float l1 = vmin(vmin(uLm, uHat - cHat), s2m);
    const float l3 = vmax(vmax(uRp, uHat + cHat), s1m);
    const float l2 = 0.5f * (l1 + l3);
    const float dl = l3 - l1;
    const float invDl = A::rcp(dl);
    const float hStarHLL = vmax((huL - huR + l3 * hR - l1 * hL) * invDl, 0.f);

    const float phiL = huL * uL + 0.5f * kGravity * hL * hL;
    const float phiR = huR * uR + 0.5f * kGravity * hR * hR;
    const float db = bR - bL;
    const float uSum = uL + uR;
    const float s1s2bar = __builtin_fmaf(0.25f, uSum * uSum, -gh);
    const float s1s2tilde = vmax(0.f, uL * uR) - gh;
    const float ct = kCriticalTol;
    const bool sonic =
        vmin(vmin(fabsf(s1s2bar), s1s2bar * s1s2tilde), s1s2bar * l1 * l3) <= ct || vmin(fabsf(l1), fabsf(l3)) < ct ||
        vmax(vmin(-l1, s1m), vmin(l3, -s2m)) > 0.f || vmin((uL + cL) * uRp, uLm * (uR - cR)) < 0.f;

    const float invBar = A::rcp(s1s2bar);
    const float dbgh = db * kGravity * (0.5f * (hL + hR));
    float ddh = sonic ? -db : dbgh * invBar;
    float ddphi = sonic ? -gh * db : -(dbgh * s1s2tilde) * invBar;
    const float hsd = hStarHLL * dl;
    const float inv13 = A::rcp(l1 * l3);
    const float dA = hsd * l1 * inv13;  // hStarHLL dl / l3
    const float dB = hsd * l3 * inv13;  // hStarHLL dl / l1
    const bool caseA = (l1 < -ct) && (l3 > ct);
    const bool subcritical = __all(caseA && !wallL && !wallR);
    if (subcritical) {
        ddh = vmax(vmin(ddh, dA), dB);
    } else {
        const bool caseB = !caseA && (l1 >= ct);
        const bool caseC = !caseA && !caseB && (l3 <= -ct);
        const float bounded = vmax(vmin(ddh, caseA ? dA : (caseB ? dB : hR)), caseA ? dB : (caseB ? -hL : dA));
        ddh = caseA || caseB || caseC ? bounded : ddh;
    }
    const float pL = -hL * db;
    const float pR = -hR * db;
    ddphi = vmax(vmin(ddphi, kGravity * vmax(pL, pR)), kGravity * vmin(pL, pR));

    const float del1 = (hR - hL) - ddh;
    const float del2 = huR - huL;
    const float del3 = (phiR - phiL) - ddphi;
    const float l1sq = l1 * l1;
    const float l3sq = l3 * l3;
    const float beta1 = (l3 * del1 - del2) * invDl;
    const float beta3 = (del2 - l1 * del1) * invDl;
    const float z1hu = beta1 * l1sq;
    const float z3hu = beta3 * l3sq;
    const float beta2 = del3 - (z1hu + z3hu);

    EdgeOut o;
    if (subcritical) {
        const float left = l2 < -kZeroTol ? 1.f : (l2 > kZeroTol ? 0.f : 0.5f);
        o.hL = beta1 * l1 + 0.f;  // the general form adds each wave to +0
        o.hR = beta3 * l3 + 0.f;
        o.huL = z1hu + __builtin_fmaf(left, beta2, 0.f);
        o.huR = __builtin_fmaf(1.f - left, beta2, 0.f) + z3hu;
        o.speed = vmax(fabsf(l1), fabsf(l3));
    } else {
        const bool kill2 = wallL || wallR;
        const float s1 = wallL ? 0.f : l1;
        const float s2 = kill2 ? 0.f : l2;
        const float s3 = wallR ? 0.f : l3;
        o = EdgeOut{0.f, 0.f, 0.f, 0.f, 0.f};
        acc_wave(s1, wallL ? 0.f : beta1 * l1, wallL ? 0.f : z1hu, o);
        acc_wave(s2, 0.f, kill2 ? 0.f : beta2, o);
        acc_wave(s3, wallR ? 0.f : beta3 * l3, wallR ? 0.f : z3hu, o);
        o.speed = vmax(fabsf(s1), fabsf(s3));
        if (dryL && dryR) o = EdgeOut{0.f, 0.f, 0.f, 0.f, 0.f};
    }
    if (anyRest && still) o = EdgeOut{0.f, 0.f, 0.f, 0.f, vmax(vmax(L.c, R.c), cHat)};
    return o;
}

}  // namespace dev
}  // namespace swe
