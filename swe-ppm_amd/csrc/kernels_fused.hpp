// kernels_fused.hpp -- flavour-U step with the previous step's update fused
// into the load ("apply on load"): one launch per time step.
//
// Launch k (k >= 1) reads Q(k-1) and the net-update sums S(k-1) of step k-1,
// forms Q(k) = update(Q(k-1), S(k-1), dt(k-1)) cell by cell as it loads them
// (dry clamp included), resolves the ghost cells of Q(k) the way
// setGhostLayer would (OUTFLOW copies, WALL negates the normal momentum,
// corners take the diagonal interior cell, other sides keep their ghosts),
// writes Q(k) to the other state buffer, then solves step k's edges from
// Q(k) and writes S(k) and the CFL maximum M(k).  dt(k-1) comes from M(k-1).
// A run of N steps is: sweep(STORE) on Q(0), N-1 fused launches, one apply.
//
// The CFL maxima rotate through three slots: launch k reads slot (k-1)%3,
// accumulates into slot k%3 and clears slot (k+1)%3, which the previous
// launch was the last to read -- so no memset is ever queued between steps.
//
// Work decomposition and edge order are those of the strip sweep
// (kernels_u.hpp), so S(k) and M(k) are bit-identical to the two-kernel step.
//
// Flavour S (V == kSplit) takes its own dt rule, update and CFL maximum through
// the same launch and keeps no quiet record.
//
// Quiet tiles.  The quiet record works on tiles of one strip (62 rows) by
// kQuietCols columns.  Launch k records per tile which of its parts had all
// four sums of every owned cell +0 (bit pattern 0) with no deferred edge --
// all its cells, its bottom and top owned rows, its first and last columns --
// and its CFL maximum, speed(k): the maximum over its x-edges on owned rows
// (those right of its columns; the left halo edge too where the tile starts a
// run of computed tiles) and its y-edges.  The tile's results depend
// only on Q(k) over its footprint: its own cells, the last column of its left
// neighbour, the first column of its right one, the top row of the tile below
// and the bottom row of the tile above (x-edge speeds count on owned rows
// only, so the corner cells of the halo feed nothing the tile reports).  If
// those parts were quiet at k-1, then Q(k) = Q(k-1) over the footprint -- an
// update by +0 sums leaves h, hu, hv bit for bit unchanged once the state has
// passed one dry clamp -- so S(k) and speed(k) repeat S(k-1) = +0 and
// speed(k-1).  If the tile was also quiet at k-2, the buffers launch k writes
// (state and sums of step k-2) already hold exactly those values.  Such a
// tile is skipped: it only carries its speed forward and adds it to the CFL
// maximum.  Launches 1 and 2 of a run never skip (their inputs may predate
// the first clamp), so every flag read was written earlier in the same run.
// Results are bit-identical with and without skipping.
//
// A wave still owns a segment of XS columns (a whole number of record
// tiles).  The skip decisions of launch k are taken by quiet_plan_kernel
// between launches k-1 and k: it carries the skipped tiles' speeds and, per
// segment with work left, lists the run of record tiles from its first to its
// last busy one (quiet tiles inside the run are recomputed, to the same
// values).  The list is compact and in domain order, per group of kPlanGroup
// segments.  Launch k then runs in list mode: wave w takes the w-th listed
// run, and waves past the count leave at once.  The busy runs thus take the
// first waves, which the dispatcher spreads over all CUs, instead of sitting
// wherever they lie in the domain (with one wave per segment in domain order,
// the CUs that hold the busy region would set the launch time while the
// others idle); with every tile busy the launch is the one without a plan.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_u.hpp"

namespace swe {

// Parts of a tile whose owned sums the quiet record tracks (one bit each):
// all cells, the bottom and top owned rows and the first and last columns --
// the halo a neighbouring tile reads.
constexpr unsigned kQuietAll = 1u, kQuietBottom = 2u, kQuietTop = 4u, kQuietLeft = 8u, kQuietRight = 16u;
// Record tiles are kQuietCols columns wide; a wave's segment of XS columns
// spans XS / kQuietCols of them.  A launch with few busy tiles lasts as long as
// one of them, whose columns are a chain of dependent operations.  us per step
// with tiles of 4 / 2 / 1 columns: 1024^2 islands 34.4 / 26.6 / 24.7, 2048^2 islands
// from the start 36.4 / 30.0 / 30.7 and from step 400 56.3 / 55.7 / 56.8, 4096^2 trench
// from the start 37.5 / 37.8 / 41.4 and from step 600 53.4 / 57.2 / 62.5, every cell
// moving 2048^2 84.8 / 85.4 / 87.6, 4096^2 301 / 301 / 313: one column solves an edge
// column twice per column and doubles the plan's work.
constexpr int kQuietCols = 2;
constexpr int kRecordWidth = 4;  // strip widths with a record are multiples of this
constexpr int kEntryBits = 4;    // list entry: segment << 2 bits | first tile << bits | tiles - 1
// Most wave segments of a block whose quiet tiles are skipped (list entries
// hold the segment in 24 bits).
constexpr long kMaxSegments = 1l << (32 - 2 * kEntryBits);
// Waves the quiet-tile plan aims to fill with busy record tiles before it
// lengthens the pieces it lists: eight per SIMD of the chip.  Measured with 4096 /
// 6144 / 8192 (us per step, strips of 8 columns at 2048^2, of 16 at 4096^2): 2048^2
// islands from step 400 61.9 / 62.3 / 55.7, every cell moving 84.5 / 84.7 / 85.4; 4096^2
// islands from step 300 102 / 92.5 / 89.0, trench from step 600 55.3 / 56.9 / 57.2.  Shorter
// pieces give more waves to hide the busy tiles' latency but solve more halo
// edges.
constexpr unsigned kPlanWaves = 8192;

// Lanes the quiet-tile plan gives a wave segment of `fine` record tiles (1 to
// 16): the smallest power of two >= fine, so that a segment's lanes share one
// wave.
__host__ __device__ constexpr int plan_lanes(int fine) {
    int l = 1;
    while (l < fine) l *= 2;
    return l;
}
// Workgroups of the plan (and entries of its count array) for nyt x nxs
// segments of `fine` record tiles.
__host__ __device__ constexpr int plan_groups(int nyt, int nxs, int fine) {
    return (nyt * nxs * plan_lanes(fine) + kPlanGroup - 1) / kPlanGroup;
}

// Waves of a launch in list mode: one per segment, or twice kPlanWaves where
// that is more (short pieces of few busy tiles), but no more than record tiles.
__host__ constexpr int list_waves(int nyt, int nxs, int nx) {
    const int tiles = nyt * ((nx + kQuietCols - 1) / kQuietCols), some = 2 * (int)kPlanWaves;
    const int want = nyt * nxs > some ? nyt * nxs : some;
    return want < tiles ? want : tiles;
}

// Which fused kernels keep the quiet record: the augmented solver's, exact
// and deferring, whose still edges give +0 sums (HLLE and f-wave leave the
// round-off of a lake at rest, so their tiles are never quiet; the in-sweep
// network variant is at its three-wave register limit and the device loop
// runs the deferring variant instead), at widths that are whole record tiles.
template <int S>
constexpr bool quiet_record(int xs) {
    return (S == SOLVER_AUGRIE || S == SOLVER_AUGRIE_DEFER) && xs % kRecordWidth == 0;
}

struct FusedIO {
    const float* h;   // Q(k-1)
    const float* hu;
    const float* hv;
    const float* b;
    float* hn;  // Q(k)
    float* hun;
    float* hvn;
    SumsView sIn;   // S(k-1)
    SumsView sOut;  // S(k)
    uint2* deferQ = nullptr;  // queue of deferred edges (SOLVER_AUGRIE_DEFER only)
    // quiet-tile record: quiet[slot * tiles + t], speed[slot * tiles + t] with
    // slot = launch index & 1 (null: no record, no skipping)
    unsigned* quiet = nullptr;
    float* speed = nullptr;
    int step = 0;  // launch index within the run (1, 2, ...)
    // list mode: workgroup g of the plan lists count[g] runs of record tiles
    // to compute at list[g * kPlanGroup ...]
    const unsigned* list = nullptr;
    const unsigned* count = nullptr;
    // >= 0: the previous update's dt, given by the caller (the per-call
    // drop-in API: updateUnknowns' dt applied on the next flux pass's load)
    float dtFixed = -1.f;
    // != 0: slotIn's maximum goes to the host under this number as the launch
    // starts (report_max).  As a launch of its own between two flux passes the
    // report took 4.4 of 29 us per call at 1000x500 and 3 of 19 at 64x50.
    unsigned rbSeq = 0u;
};

// The w-th list entry, or kNoEntry past the last one.  Each lane takes four
// group counts (a block of 4096 x 4096 has 134 groups), a scan over the wave
// finds the lane whose groups hold the entry, and the rest is scalar.
constexpr unsigned kNoEntry = 0xffffffffu;  // no entry: first tile + tiles - 1 < tiles per segment
__device__ __forceinline__ unsigned listed_item(const FusedIO& io, int groups, int w) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < groups; base += 256) {  // uniform per wave
        unsigned c[4], sum = 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int g = base + 4 * lane + i;
            c[i] = g < groups ? io.count[g] : 0u;
            sum += c[i];
        }
        const unsigned incl = wave_scan(sum);
        const unsigned total = (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
        if ((unsigned)w < total) {
            const int l = __builtin_ctzll(__ballot(incl > (unsigned)w));
            int g = base + 4 * l;
            unsigned at = (unsigned)w - (unsigned)__builtin_amdgcn_readlane((int)(incl - sum), l);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const unsigned ci = (unsigned)__builtin_amdgcn_readlane((int)c[i], l);
                if (at < ci) break;
                at -= ci;
                ++g;
            }
            return io.list[(size_t)g * kPlanGroup + at];
        }
        w -= (int)total;
    }
    return kNoEntry;
}

struct Q3 {
    float h, hu, hv;
};

__device__ __forceinline__ bool is_ow(int t) { return t == OUTFLOW || t == WALL; }

template <int S, int XS, int V>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(fused_waves_per_simd(S), 8))) void fused_u_kernel(
    StateView v, FusedIO io, BoundaryInfo bi, DeviceCtl* ctl, int slotIn, int slotOut, int slotClear, float* dtLog,
    int logIdx) {
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6));
    const int nyt = (v.ny + kStripRows - 1) / kStripRows;
    const int nxs = (v.nx + XS - 1) / XS;
    const int nx = v.nx, ny = v.ny;

    float dt = io.dtFixed;
    if (!(dt >= 0.f)) {
        const float s = ctl->smax[slotIn].value();
        dt = V == kSplit ? split_timestep(s, v.dx) : timestep_from_max(s, v.dx, v.dy);
    }
    if (blockIdx.x == 0) {
        ctl->smax[slotClear].clear();
        if (threadIdx.x == 0) {
            if (io.rbSeq != 0u) report_max(ctl, slotIn, io.rbSeq);
            ctl->defer[slotClear] = 0u;
            ctl->busy[slotClear] = 0u;
            ctl->dt = dt;
            ctl->t += dt;
            ctl->steps += 1;
            if (dtLog) dtLog[logIdx] = dt;
        }
    }
    constexpr bool kRecord = V != kSplit && quiet_record<S>(XS);
    const int items = nyt * nxs;
    // list mode: entry after entry until the list ends (the grid covers the
    // usual lists once)
    for (int w = wave;; w += gridDim.x * kWavesPerGroup) {
        int item = w, first = 0, ncols = XS;
        if (kRecord && io.list) {
            const unsigned e =
                __builtin_amdgcn_readfirstlane(listed_item(io, plan_groups(nyt, nxs, XS / kQuietCols), w));
            if (e == kNoEntry) return;  // uniform per wave
            constexpr unsigned mask = (1u << kEntryBits) - 1u;
            item = (int)(e >> (2 * kEntryBits));
            first = (int)((e >> kEntryBits) & mask);
            ncols = (int)((e & mask) + 1u) * kQuietCols;
        }
        if (item >= items) return;  // uniform per wave
        const int yt = item % nyt;
        const int xs = item / nyt;
        const int slotNow = (io.step & 1) * nyt * ((nx + kQuietCols - 1) / kQuietCols);
        const dev::SolverCtx<S> solver(S == SOLVER_AUGRIE_MLP ? ctl->mlp : nullptr);

        const float dtdx = dt / v.dx;
        const float dtdy = dt / v.dy;
        const int x0 = 1 + xs * XS + first * kQuietCols;
        const int x1 = min(x0 + ncols - 1, nx);
        const bool ghostRows = yt == 0 || kStripRows * yt + 63 >= ny + 1;  // the strip holds a ghost row
        const int tB = bi.type[BND_BOTTOM], tT = bi.type[BND_TOP], tL = bi.type[BND_LEFT], tR = bi.type[BND_RIGHT];

        auto tile = [&](auto form, int lane) -> bool {
            constexpr bool N = decltype(form)::value;
            using A = CellMath<N>;
            const int y = kStripRows * yt + lane;
            const bool rowValid = y <= ny + 1;
            const int yc = rowValid ? y : ny + 1;
            const bool owned = (lane >= 1) && (lane <= kStripRows) && (y <= ny);
            const bool rowInterior = (y >= 1) && (y <= ny);
            const bool hEdgeValid = (lane <= kStripRows) && (y <= ny);
            const bool rowBottom = (y == 0);
            const bool rowTop = (y == ny + 1);
            const bool carryRow = owned || (rowBottom && lane == 0) || (rowTop && lane >= 1);

            // a column as stored: Q(k-1), S(k-1) and the bed (past the tile its right halo
            // column again, which the caches hold: 2048^2 moving 75.0 -> 73.7 us per
            // launch, Hybrid 1500 x 901 39.5 -> 38.6)
            struct Raw {
                float h, hu, hv, sx, sy, su, sv, b;
            };
            auto load_raw = [&](int x) -> Raw {
                const size_t c = (size_t)min(x, x1 + 1) * v.pitch;
                const unsigned rc = lane_bytes(yc);
                return Raw{col_get(io.h, c, rc),      col_get(io.hu, c, rc),     col_get(io.hv, c, rc),
                           col_get(io.sIn.sx, c, rc), col_get(io.sIn.sy, c, rc), col_get(io.sIn.su, c, rc),
                           col_get(io.sIn.sv, c, rc), col_get(v.b, c, rc)};
            };
            // Q(k) of its cells: interior cells updated, ghosts as stored
            auto updated = [&](const Raw& r, int x) -> Q3 {
                Q3 q{r.h, r.hu, r.hv};
                if (x >= 1 && x <= nx && rowInterior) {
                    const Cell u = step_cell<V>(q.h, q.hu, q.hv, dtdx, dtdy, r.sx, r.sy, r.su, r.sv);
                    q = Q3{u.h, u.hu, u.hv};
                }
                return q;
            };
            // ghost rows of an interior column: the boundary value of the row next to
            // it (lane+1 for the bottom row, lane-1 for the top row)
            auto fix_rows = [&](Q3 q) -> Q3 {
                if (!ghostRows) return q;
                const float dh = __shfl_down(q.h, 1, 64), dhu = __shfl_down(q.hu, 1, 64), dhv = __shfl_down(q.hv, 1, 64);
                const float uh = __shfl_up(q.h, 1, 64), uhu = __shfl_up(q.hu, 1, 64), uhv = __shfl_up(q.hv, 1, 64);
                if (rowBottom && is_ow(tB)) q = Q3{dh, dhu, (tB == WALL) ? -dhv : dhv};
                if (rowTop && is_ow(tT)) q = Q3{uh, uhu, (tT == WALL) ? -uhv : uhv};
                return q;
            };
            // a ghost column next to the interior column value `in` (same lane);
            // corners take the diagonal interior cell (from the neighbouring lane)
            auto fix_column = [&](Q3 raw, Q3 in, int type) -> Q3 {
                const float dh = __shfl_down(in.h, 1, 64), dhu = __shfl_down(in.hu, 1, 64), dhv = __shfl_down(in.hv, 1, 64);
                const float uh = __shfl_up(in.h, 1, 64), uhu = __shfl_up(in.hu, 1, 64), uhv = __shfl_up(in.hv, 1, 64);
                Q3 q = raw;
                if (rowInterior && is_ow(type)) q = Q3{in.h, (type == WALL) ? -in.hu : in.hu, in.hv};
                if (rowBottom) q = Q3{dh, dhu, dhv};
                if (rowTop) q = Q3{uh, uhu, uhv};
                return q;
            };
            auto store = [&](int x, const Q3& q) {
                const size_t c = (size_t)x * v.pitch;
                const unsigned ry = lane_bytes(y);
                col_set(io.hn, c, ry, q.h);
                col_set(io.hun, c, ry, q.hu);
                col_set(io.hvn, c, ry, q.hv);
            };

            // columns x0-1, x0 and (a software pipeline) x0+1: every load at once.
            // The learned middle state loads column by column: its network call and
            // the deferring sweep's seven waves leave no registers to load ahead.
            constexpr bool kAhead = S != SOLVER_AUGRIE_MLP && S != SOLVER_AUGRIE_DEFER;
            const Raw r0 = load_raw(x0 - 1), r1 = load_raw(x0);
            Raw ahead{};
            if constexpr (kAhead) ahead = load_raw(x0 + 1);
            Q3 cur = fix_rows(updated(r1, x0));
            Q3 prev = updated(r0, x0 - 1);
            if (x0 == 1) prev = fix_column(prev, cur, tL);
            if (x0 == 1 && carryRow) store(0, prev);

            const CellQ pq = cell_q<A>(prev.h, prev.hu, prev.hv, r0.b);
            CellQ cq = cell_q<A>(cur.h, cur.hu, cur.hv, r1.b);
            bool outside = outside_range<N>(pq) || outside_range<N>(cq);
            dev::EdgeOut e = solver.template solve<A>(pq.xside(), cq.xside());
            // record tile of the columns being solved: a deferred edge touching it
            // makes it not quiet; the halo edge (x0-1 | x0) counts for the first
            bool loud = false;
            if constexpr (S == SOLVER_AUGRIE_DEFER) {
                loud = e.speed < 0.f;
                e = defer_edge(e, owned && x0 == 1, make_uint2(0u, (unsigned)y), io.deferQ, &ctl->defer[slotOut]);
            }
            float carryH = e.hR, carryHu = e.huR;
            // The x- and the y-edges' maxima of this lane's row in the record tile.
            // x-edges count on owned rows (each interior row is owned by one strip),
            // so a record tile's maximum depends on its footprint only; which lanes
            // count is the same in every column, so they are masked at the tile's end.
            // Flavour S counts the x-edges of every row: edge (0 | 1) by the
            // first segment, any other halo edge by the segment left of it (the column
            // loaded as halo lacks its ghost rows' boundary condition, as do lanes past
            // the top ghost row).
            float smaxX = V != kSplit ? e.speed : x0 == 1 ? dev::smax(0.f, e.speed) : 0.f, smaxY = 0.f;
            auto tile_max = [&] {
                if constexpr (V == kSplit) return wave_max<N>(rowValid ? smaxX : 0.f);
                return wave_max<N>(dev::smax(owned ? smaxX : 0.f, hEdgeValid ? smaxY : 0.f));
            };
            // the segment's maximum over its record tiles, wave-uniform (float bits:
            // non-negative floats order like unsigned integers)
            unsigned smaxRun = 0u;
            // lanes whose owned sums were not all +0 in some column of the record
            // tile, and in its first and last column
            unsigned long long loudAll = 0u, loudFirst = 0u, loudLast = 0u;

            for (int x = x0; x <= x1; ++x) {
                // column x+1 of Q(k); the loads of the next one overlap this one's edges
                const Raw r = kAhead ? ahead : load_raw(x + 1);
                if constexpr (kAhead) ahead = load_raw(x + 2);
                Q3 nxt = fix_rows(updated(r, x + 1));
                if (x + 1 == nx + 1) nxt = fix_column(nxt, cur, tR);
                const CellQ nq = cell_q<A>(nxt.h, nxt.hu, nxt.hv, r.b);
                outside = outside || outside_range<N>(nq);

                if (carryRow) store(x, cur);
                if (x + 1 == nx + 1 && carryRow) store(nx + 1, nxt);

                dev::EdgeOut ev = solver.template solve<A>(cq.xside(), nq.xside());
                bool loudEdge = false;
                if constexpr (S == SOLVER_AUGRIE_DEFER) {
                    loudEdge = ev.speed < 0.f;
                    ev = defer_edge(ev, owned, make_uint2((unsigned)x, (unsigned)y), io.deferQ, &ctl->defer[slotOut]);
                }
                smaxX = A::max(smaxX, ev.speed);
                dev::EdgeOut eh = solver.template solve<A>(cq.yside(), cq.yside_from_lane_above());
                if constexpr (S == SOLVER_AUGRIE_DEFER) {
                    loud = loud || loudEdge || eh.speed < 0.f;
                    eh = defer_edge(eh, owned || y == 0, make_uint2((unsigned)x | kDeferY, (unsigned)y), io.deferQ,
                                    &ctl->defer[slotOut]);
                }
                if constexpr (V != kSplit) smaxY = A::max(smaxY, eh.speed);
                const float aH = __shfl_up(eh.hR, 1, 64);
                const float aHv = __shfl_up(eh.huR, 1, 64);
                const float sx = carryH + ev.hL, su = carryHu + ev.huL, sy = aH + eh.hL, sv = aHv + eh.huL;
                if (owned) {
                    const size_t c = (size_t)x * v.pitch;
                    const unsigned ry = lane_bytes(y);
                    col_set(io.sOut.sx, c, ry, sx);
                    col_set(io.sOut.su, c, ry, su);
                    col_set(io.sOut.sy, c, ry, sy);
                    col_set(io.sOut.sv, c, ry, sv);
                }
                if constexpr (kRecord) {
                    const bool nonzero =
                        (__float_as_uint(sx) | __float_as_uint(su) | __float_as_uint(sy) | __float_as_uint(sv)) != 0u;
                    loudLast = __ballot(owned && nonzero);
                    loudAll |= loudLast;
                    if (((x - 1) & (kQuietCols - 1)) == 0) loudFirst = loudLast;
                }
                carryH = ev.hR;
                carryHu = ev.huR;
                cur = nxt;
                cq = nq;
                // the end of a record tile: its parts' flags and its maximum.  A tile
                // reports its right edge (x | x+1) and, first in a run, its left halo
                // edge; the tile of column 1 always starts a run, so every x-edge is
                // in some record, and each record's edges lie in its tile's footprint.
                // A deferred edge at the boundary touches both tiles.
                if (kRecord && ((x & (kQuietCols - 1)) == 0 || x == x1)) {  // uniform per wave
                    const float tileMax = tile_max();
                    smaxRun = max(smaxRun, __builtin_amdgcn_readfirstlane(__float_as_uint(tileMax)));
                    if (io.quiet) {
                        unsigned quiet = (loudAll == 0u ? kQuietAll : 0u) |
                                         ((loudAll >> 1 & 1u) == 0u ? kQuietBottom : 0u) |
                                         ((loudAll >> kStripRows & 1u) == 0u ? kQuietTop : 0u) |
                                         (loudFirst == 0u ? kQuietLeft : 0u) | (loudLast == 0u ? kQuietRight : 0u);
                        if (__any(loud)) quiet = 0u;
                        if (lane == 0) {
                            const int rec = slotNow + yt + nyt * ((x - 1) / kQuietCols);
                            io.quiet[rec] = quiet;
                            io.speed[rec] = tileMax;
                        }
                    }
                    smaxX = smaxY = 0.f;
                    loud = loudEdge;
                    loudAll = loudFirst = 0u;
                }
            }

            if (N && __any(outside)) return false;
            if constexpr (!kRecord) smaxRun = __float_as_uint(tile_max());
            if (lane == 0) raise_max(ctl->smax[slotOut], smaxRun);
            return true;
        };
        run_tile<dev::SolverCtx<S>, V>(threadIdx.x & 63, tile);
        if (!(kRecord && io.list)) return;
    }
}

}  // namespace swe
