// edge_solver.hpp -- one edge with any solver, in the form that its cells allow:
// the general one (solvers_dev.hpp) or the short one for cells in
// in_normal_range (exact_math.hpp, augrie_normal.hpp).
#pragma once

#include "augrie_normal.hpp"
#include "exact_math.hpp"
#include "solvers_dev.hpp"

namespace swe {
namespace dev {

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

// One edge with solver S, in the general form or (A = NormalRange) the short
// one; the results are the same.
template <int S, class A = Ieee>
__device__ __forceinline__ EdgeOut solve_edge(const Side& L, const Side& R) {
    if constexpr (S == SOLVER_FWAVE) return fwave<A>(L, R);
    if constexpr (S == SOLVER_HLLE) return hlle<A>(L, R);
    if constexpr (S == SOLVER_HYBRID)
        if (L.h >= kHybridTol && R.h >= kHybridTol) return fwave<A>(L, R);
    if constexpr (S == SOLVER_AUGRIE || S == SOLVER_HYBRID) {
        if constexpr (A::kNormal)
            return augrie_normal(L, R);
        else
            return augrie(L, R);
    }
}

// The speed alone that solver S reports for an edge (the light solvers; Hybrid
// takes the augmented solver's from its whole edge, on the few shallow lanes).
template <int S, class A>
__device__ __forceinline__ float solver_speed(const Side& L, const Side& R) {
    if constexpr (S == SOLVER_HYBRID) {
        float speed = edge_speed<SOLVER_FWAVE, A>(L, R);
        if (!(L.h >= kHybridTol && R.h >= kHybridTol)) speed = solve_edge<SOLVER_AUGRIE, A>(L, R).speed;
        return speed;
    } else {
        return edge_speed<S, A>(L, R);
    }
}

// Solver with per-kernel state, built once at kernel start from an optional
// parameter block (the learned middle state keeps its network weights in
// registers; the exact solvers have no state).  kNormalForm: the sweeps solve
// the edges of ordinary cells in the short form (run_tile in kernels_u.hpp).
template <int S>
struct SolverCtx {
    static constexpr bool kNormalForm = true;
    __device__ __forceinline__ explicit SolverCtx(const unsigned*) {}
    template <class A = Ieee>
    __device__ __forceinline__ EdgeOut solve(const Side& L, const Side& R) const {
        return solve_edge<S, A>(L, R);
    }
};

// Convenience for raw edge states (one-off evaluations).
template <int S, class A = Ieee>
__device__ __forceinline__ EdgeOut solve_raw(float hL, float hR, float huL, float huR, float bL, float bR) {
    return solve_edge<S, A>(cell_side<A>(hL, huL, bL), cell_side<A>(hR, huR, bR));
}

}  // namespace dev
}  // namespace swe
