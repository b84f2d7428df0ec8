// kernels_advance.hpp -- flavour-U step of the light solvers (HLLE, f-wave, and on
// larger blocks Hybrid) in one pass over the state: one launch per time step, no sums in memory.
//
// Launch k reads Q(k) (ghost cells as setGhostLayer leaves them) and M(k), the
// CFL maximum of its edges, solves the edges of Q(k), updates the cells with
// dt(k) from M(k), writes Q(k+1) to the other buffer (ghost cells of OUTFLOW /
// WALL sides and corners derived from it) and reduces M(k+1), the maximum over
// the edges of Q(k+1), whose speeds take a root and a division per edge.  A run of N
// steps is a max sweep of Q(0) and N of these launches; the last one leaves
// the ghost cells as Q(N-1)'s and reduces nothing.
//
// What it trades: it moves 28 bytes per cell (h, hu, hv, b read, h, hu, hv
// written) against the fused step's 60 (four sums written and read besides),
// and solves the speeds of every edge a second time.  The light solvers are
// bound by memory, so that pays where the state and sums do not stay in the
// caches near the SIMDs (advance_pays); the augmented solver keeps its sums, whose
// zeros are the record that lets quiet tiles be skipped.
//
// Work decomposition: the strip sweep's, with a deeper halo.  A wave owns 61
// rows (lanes 1..61); lane 62 updates the row above too, for the speed of the
// edge between them, and lanes 0 and 63 hold its neighbours.  Along x it owns XS
// columns and also updates the one before them, for the speed of the edge
// between that column and its first.  Measured, 40 steps of HLLE on 4096^2: 141 us
// per launch against 292 for the fused step, of which vector issue takes most; a
// copy of the 28 bytes per cell takes 92.  Every sum, update and speed is formed by
// the same operations as in the other strategies, and the maximum does not
// depend on the order: results are bit-identical.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_fused.hpp"

namespace swe {

constexpr int kAdvanceRows = 61;  // owned rows per wavefront

template <int S, int XS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(fused_waves_per_simd(S), 8))) void
advance_u_kernel(StateView v, float* hn, float* hun, float* hvn, BoundaryInfo bi, DeviceCtl* ctl, int slotIn,
                 int slotOut, int slotClear, int last, float* dtLog, int logIdx) {
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6));
    const int nx = v.nx, ny = v.ny;
    const int nyt = (ny + kAdvanceRows - 1) / kAdvanceRows;
    const int nxs = (nx + XS - 1) / XS;
    const float dt = timestep_from_max(ctl->smax[slotIn].value(), v.dx, v.dy);
    if (blockIdx.x == 0) ctl->smax[slotClear].clear();
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl->dt = dt;
        ctl->t += dt;
        ctl->steps += 1;
        if (dtLog) dtLog[logIdx] = dt;
    }
    if (wave >= nyt * nxs) return;  // uniform per wave
    const dev::SolverCtx<S> solver(nullptr);
    const int yt = wave % nyt;
    const int xs = wave / nyt;
    const float dtdx = dt / v.dx;
    const float dtdy = dt / v.dy;
    const int x0 = 1 + xs * XS;
    const int x1 = min(x0 + XS - 1, nx);
    const int xa = max(x0 - 1, 1);  // first column updated
    const bool ghostRows = yt == 0 || kAdvanceRows * yt + 63 >= ny + 1;  // the strip holds a ghost row
    const int tB = bi.type[BND_BOTTOM], tT = bi.type[BND_TOP], tL = bi.type[BND_LEFT], tR = bi.type[BND_RIGHT];

    auto tile = [&](auto form, int lane) -> bool {
        constexpr bool N = decltype(form)::value;
        using A = CellMath<N>;
        const int y = kAdvanceRows * yt + lane;
        const int yc = min(y, ny + 1);
        const bool owned = (lane >= 1) && (lane <= kAdvanceRows) && (y <= ny);
        const bool interior = (y >= 1) && (y <= ny);
        const bool rowBottom = (y == 0);
        const bool rowTop = (y == ny + 1);
        // rows this wave writes; the top ghost row belongs to the strip of row ny
        const bool writeRow = owned || rowBottom || (rowTop && lane >= 2 && lane <= kAdvanceRows + 1);
        const bool hEdge = owned || rowBottom;  // this lane's edge (y | y+1) counts

        auto load = [&](int x) -> Q3 {
            const size_t c = (size_t)x * v.pitch;
            const unsigned r = lane_bytes(yc);
            return Q3{col_get(v.h, c, r), col_get(v.hu, c, r), col_get(v.hv, c, r)};
        };
        auto bed = [&](int x) { return col_get(v.b, (size_t)x * v.pitch, lane_bytes(yc)); };
        const unsigned rowBytes = writeRow ? (unsigned)y * 4u : kNoStore;
        auto store = [&](int x, unsigned bytes, const Q3& q) {
            const size_t c = (size_t)x * v.pitch;
            col_put(hn, c, v.pitch, bytes, q.h);
            col_put(hun, c, v.pitch, bytes, q.hu);
            col_put(hvn, c, v.pitch, bytes, q.hv);
        };
        // Q(k+1)'s ghost column next to the updated interior column `in`
        // (corners: the diagonal interior cell, from the neighbouring lane)
        auto ghost_column = [&](Q3 raw, Q3 in, int type) -> Q3 {
            const float dh = __shfl_down(in.h, 1, 64), dhu = __shfl_down(in.hu, 1, 64), dhv = __shfl_down(in.hv, 1, 64);
            const float uh = __shfl_up(in.h, 1, 64), uhu = __shfl_up(in.hu, 1, 64), uhv = __shfl_up(in.hv, 1, 64);
            Q3 q = raw;
            if (last) return q;
            if (interior && is_ow(type)) q = Q3{in.h, (type == WALL) ? -in.hu : in.hu, in.hv};
            if (rowBottom) q = Q3{dh, dhu, dhv};
            if (rowTop) q = Q3{uh, uhu, uhv};
            return q;
        };

        const Q3 left = load(xa - 1);
        const float leftB = bed(xa - 1);
        Q3 cur = load(xa);
        const CellQ pq = cell_q<A>(left.h, left.hu, left.hv, leftB);
        CellQ cq = cell_q<A>(cur.h, cur.hu, cur.hv, bed(xa));
        bool outside = outside_range<N>(pq) || outside_range<N>(cq);
        const dev::EdgeOut e = solver.template solve<A>(pq.xside(), cq.xside());
        float carryH = e.hR, carryHu = e.huR;
        Q3 ahead = load(xa + 1);
        float aheadB = bed(xa + 1);
        // (the loop's first wait counts as many stores behind the loads as later ones)
        store(xa, kNoStore, cur);
        CellQ wq = cq;  // Q(k+1) of the column before x
        // the x- and y-edges' maxima of this lane's row; which lanes count is the
        // same for every column, so they are masked once, at the end
        float smaxX = 0.f, smaxY = 0.f;
        for (int x = xa; x <= x1; ++x) {
            // column x+1 of Q(k); the one after it is loaded meanwhile (column
            // nx + 1 at most, not used past x1 + 1)
            const Q3 nxt = ahead;
            const CellQ nq = cell_q<A>(nxt.h, nxt.hu, nxt.hv, aheadB);
            const int xn = min(x + 2, nx + 1);
            ahead = load(xn);
            aheadB = bed(xn);
            outside = outside || outside_range<N>(nq);
            const dev::EdgeOut ev = solver.template solve<A>(cq.xside(), nq.xside());
            const dev::EdgeOut eh = solver.template solve<A>(cq.yside(), cq.yside_from_lane_above());
            const float aH = __shfl_up(eh.hR, 1, 64);
            const float aHv = __shfl_up(eh.huR, 1, 64);
            Q3 q{cq.h, cq.hu, cq.hv};
            if (interior) {
                const Cell u = update_cell(cq.h, cq.hu, cq.hv, dtdx, dtdy, carryH + ev.hL, aH + eh.hL, carryHu + ev.huL,
                                           aHv + eh.huL);
                q = Q3{u.h, u.hu, u.hv};
            }
            carryH = ev.hR;
            carryHu = ev.huR;
            if (ghostRows && !last) {
                const float dh = __shfl_down(q.h, 1, 64), dhu = __shfl_down(q.hu, 1, 64), dhv = __shfl_down(q.hv, 1, 64);
                const float uh = __shfl_up(q.h, 1, 64), uhu = __shfl_up(q.hu, 1, 64), uhv = __shfl_up(q.hv, 1, 64);
                if (rowBottom && is_ow(tB)) q = Q3{dh, dhu, (tB == WALL) ? -dhv : dhv};
                if (rowTop && is_ow(tT)) q = Q3{uh, uhu, (tT == WALL) ? -uhv : uhv};
            }
            const bool mine = x >= x0;
            store(x, mine ? rowBytes : kNoStore, q);
            Q3 edge{0.f, 0.f, 0.f};  // Q(k+1) of ghost column 0 or nx + 1
            if (x == 1) {
                edge = ghost_column(left, q, tL);
                store(0, rowBytes, edge);
                wq = cell_q<A>(edge.h, edge.hu, edge.hv, leftB);
            }
            if (!last) {
                const CellQ uq = cell_q<A>(q.h, q.hu, q.hv, cq.b);
                outside = outside || outside_range<N>(uq);
                if (mine) {  // uniform; column x0 - 1 only lends its right edge
                    smaxX = A::max(smaxX, dev::solver_speed<S, A>(wq.xside(), uq.xside()));
                    smaxY = A::max(smaxY, dev::solver_speed<S, A>(uq.yside(), uq.yside_from_lane_above()));
                }
                wq = uq;
            }
            if (x == nx) {
                edge = ghost_column(nxt, q, tR);
                store(nx + 1, rowBytes, edge);
                if (!last) {
                    const CellQ rq = cell_q<A>(edge.h, edge.hu, edge.hv, nq.b);
                    outside = outside || outside_range<N>(rq);
                    smaxX = A::max(smaxX, dev::solver_speed<S, A>(wq.xside(), rq.xside()));
                }
            }
            cq = nq;
        }
        if (N && __any(outside)) return false;
        if (!last) {
            const float smaxv = wave_max<N>(dev::smax(owned ? smaxX : 0.f, hEdge ? smaxY : 0.f));
            if (lane == 0) raise_max(ctl->smax[slotOut], __float_as_uint(smaxv));
        }
        return true;
    };
    run_tile<dev::SolverCtx<S>, 0>(threadIdx.x & 63, tile);
}

}  // namespace swe
