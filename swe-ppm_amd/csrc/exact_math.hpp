// exact_math.hpp -- division and square root of the solvers: the same
// correctly rounded single-precision results in two forms.
//
//   Ieee         the compiler's forms, for every operand.  A division costs 10
//                VALU instructions (operand scaling, one quarter-rate
//                reciprocal, refinement, the fix-up of special operands), a
//                square root 15 (scaling, the hardware root, a test of both
//                neighbours, special operands).
//   NormalRange  for operands whose quotients, roots and residuals are normal
//                numbers: no scaling, no special operands.  A reciprocal is 3
//                instructions, a division 6, a square root 5.
//
// Why NormalRange rounds correctly:
//   reciprocal   v_rcp_f32 and one Newton step with a fused residual,
//                y' = y + y (1 - b y).  On gfx950 it equals RN(1 / b) for every
//                b with 2^-126 <= b < 2^126 (all 2^31 positive floats
//                compared with the IEEE division).
//   division     q0 = RN(a y') with the reciprocal above, the fused residual
//                r = a - b q0 and q = RN(q0 + r y') (Markstein 1990, IBM J. Res.
//                Dev. 34).  On gfx950 all 2^46 pairs of mantissas give RN(a / b)
//                (checked through the exact residual in double precision);
//                exponents only scale it while a, q and r stay normal, which
//                |a| >= 2^-102, 2^-126 <= b < 2^126 and a normal quotient give.
//   square root  v_rsq_f32, g = x y, and one step with the fused residual,
//                g + (x - g^2) y / 2: equals RN(sqrt(x)) for every x with
//                2^-102 <= x <= FLT_MAX on gfx950 (all of them compared).
// Zero: a zero numerator gives +0 (an IEEE division keeps the sign); sqrt0 also
// takes x = 0.  A numerator below 2^-102 may be rounded wrongly, by less than
// 2^-100 of 1 / b; the callers add such quotients to numbers far larger
// (in_normal_range).
#pragma once

#include <hip/hip_runtime.h>

namespace swe {
namespace dev {

struct Ieee {
    static constexpr bool kNormal = false;
    __device__ __forceinline__ static float rcp(float b) { return 1.f / b; }
    __device__ __forceinline__ static float div(float a, float b) { return a / b; }
    __device__ __forceinline__ static float sqrt(float x) { return sqrtf(x); }
    // std::min / std::max semantics (first operand wins ties), not fminf / fmaxf
    __device__ __forceinline__ static float min(float a, float b) { return (b < a) ? b : a; }
    __device__ __forceinline__ static float max(float a, float b) { return (a < b) ? b : a; }
};

struct NormalRange {
    static constexpr bool kNormal = true;
    __device__ __forceinline__ static float rcp(float b) {
        const float y = __builtin_amdgcn_rcpf(b);
        return __builtin_fmaf(__builtin_fmaf(-b, y, 1.f), y, y);
    }
    __device__ __forceinline__ static float div(float a, float b) {
        const float y = rcp(b);
        const float q = a * y;
        return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
    }
    __device__ __forceinline__ static float root(float x, float y) {
        const float g = x * y;
        return __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
    }
    __device__ __forceinline__ static float sqrt(float x) { return root(x, __builtin_amdgcn_rsqf(x)); }
    // one instruction, for results of arithmetic that are no NaN (the sign of a
    // zero may differ from Ieee's)
    __device__ __forceinline__ static float min(float a, float b) { return __builtin_fminf(a, b); }
    __device__ __forceinline__ static float max(float a, float b) { return __builtin_fmaxf(a, b); }
    // x = 0 too: the reciprocal root of a positive number keeps 0 * y at 0
    __device__ __forceinline__ static float sqrt0(float x) {
        return root(x, __builtin_amdgcn_rsqf(__builtin_fmaxf(x, 0x1p-100f)));
    }
};

}  // namespace dev
}  // namespace swe
