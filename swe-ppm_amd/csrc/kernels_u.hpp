// kernels_u.hpp -- flavour-U step kernels (every edge from one state, unsplit
// update with dry clamp), the step of all of the reference's parallel blocks
// (src/blocks/SWE_DimensionalSplittingMpi.cpp:383-518).
//
// Data layout in HBM: each field is one column-major array like the
// reference's Float2D (a[x][y] at x*pitch + y, y contiguous), so a wavefront
// reads 64 consecutive y at one x: one 256-byte coalesced load per field.
//
// Work decomposition ("strip"): one wavefront owns 62 consecutive rows
// y0..y0+61 (lanes 1..62; lane 0 and lane 63 hold the rows just below and
// above) and marches along x over a segment of XS columns.  At column x a
// lane holds cell (x, y) and loads cell (x+1, y):
//   * the vertical edge (x | x+1) is solved in-lane; its right-going part is
//     carried in registers to the next column;
//   * the horizontal edge (y | y+1) takes the upper cell from lane+1 with a
//     cross-lane shuffle; the up-going part of edge (y-1 | y) comes back from
//     lane-1 the same way.
// Each interior edge is solved once per strip (plus one halo x-edge per
// segment), net updates never leave registers, and the CFL maximum is
// reduced in-wave; a wave raises its die's word of it only where its own is
// larger (raise_max).
//
// Modes:
//   MODE_MAX    edges -> max speed only (first half of the two-pass step);
//   MODE_STORE  edges -> per-cell net-update sums (4 floats) + max speed;
//   MODE_UPDATE edges -> update with dt from the device max, written to the
//               other state buffer (second half of the two-pass step).
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <type_traits>

#include "mlp.hpp"
#include "edge_solver.hpp"
#include "swe_common.h"

namespace swe {

enum SweepMode : int { MODE_MAX = 0, MODE_STORE = 1, MODE_UPDATE = 2 };

constexpr int kStripRows = 62;  // owned rows per wavefront
constexpr int kWavesPerGroup = 4;
constexpr int kPlanGroup = 1024;  // wave segments per workgroup of the quiet-tile plan

// ---- strip tiles of the batched engine --------------------------------------
// The strips of kStripRows rows below a block's last strip are cut into
// column segments of XS columns, one wave per (strip, segment).  The last
// strip (the tail, R = ny - kStripRows * (nyt - 1) rows) follows: when R is
// small, its inner segments (full XS columns, away from the left and right
// boundary columns) share waves, `pack` segments per wave, each on a group of
// R + 2 lanes (R rows with a halo lane on either side) laid side by side.
// Every lane computes what the lane of an unpacked strip computes for its row
// and column, so the packing does not change any result.  (The single-block
// kernels keep one wave per (strip, segment): on a large block the tail is a
// small share of the waves, and its clamped lanes make those waves cheap.)
struct StripTiling {
    int nyt, nxs, pack, items;
};

__host__ __device__ inline StripTiling strip_tiling(int nx, int ny, int xs) {
    StripTiling g;
    g.nyt = (ny + kStripRows - 1) / kStripRows;
    g.nxs = (nx + xs - 1) / xs;
    const int perWave = 64 / (ny - kStripRows * (g.nyt - 1) + 2);
    g.pack = (perWave >= 2 && g.nxs >= 4) ? perWave : 1;
    g.items = (g.nyt - 1) * g.nxs + (g.pack == 1 ? g.nxs : 2 + (g.nxs - 2 + g.pack - 1) / g.pack);
    return g;
}

struct TileLanes {
    int yt;            // strip (uniform)
    int xs0;           // first column segment of the item (uniform)
    int xs;            // column segment of this lane's group
    int r;             // row of the lane in the strip: 0 and R+1 are halo rows; 63 on idle lanes
    bool first, last;  // the item's segments are the block's first / last (uniform)
};

// item `tile` of a block's strip tiling: order (strip, segment) with the
// strip fastest below the tail, then the tail's first and last segments,
// then its packed inner segments
__device__ __forceinline__ TileLanes tile_lanes(int nyt, int nxs, int pack, int ny, int tile, int lane) {
    TileLanes t;
    const int body = (nyt - 1) * nxs;
    int lanesPerGroup = 64, groups = 1;
    if (tile < body) {
        t.yt = tile % (nyt - 1);
        t.xs0 = tile / (nyt - 1);
    } else {
        const int u = tile - body;
        t.yt = nyt - 1;
        if (pack == 1) {
            t.xs0 = u;
        } else if (u < 2) {
            t.xs0 = u ? nxs - 1 : 0;
        } else {
            t.xs0 = 1 + (u - 2) * pack;
            groups = min(pack, nxs - 1 - t.xs0);
            lanesPerGroup = ny - kStripRows * t.yt + 2;
        }
    }
    const int g = lane / lanesPerGroup;
    t.xs = t.xs0 + g;
    t.r = lane - g * lanesPerGroup;
    if (g >= groups) {
        t.xs = t.xs0;
        t.r = 63;
    }
    t.first = t.xs0 == 0;
    t.last = t.xs0 == nxs - 1;
    return t;
}

// columns of every segment of the item: XS, fewer for the last
__device__ __forceinline__ int tile_columns(const TileLanes& t, int nx, int xs) {
    return min(xs, nx - t.xs0 * xs);
}

struct StateView {
    float* h;
    float* hu;
    float* hv;
    const float* b;
    int nx, ny, pitch;
    float dx, dy;
};

struct SumsView {  // per-cell net-update sums, same layout as the state
    float* sx;     // h, x-edges:  R(x-1|x) + L(x|x+1)
    float* sy;     // h, y-edges:  A(y-1|y) + B(y|y+1)
    float* su;     // hu, x-edges
    float* sv;     // hv, y-edges
};

struct BoundaryInfo {
    int type[4];  // BoundaryType per side
};

// A CFL maximum (float bits of non-negative speeds: unsigned order == float
// order), kept in kCflWords words, one to a cache line: workgroup g raises word
// g % kCflWords, and the maximum is that over the words.  Consecutive
// workgroups go to the chip's dies in turn, so a word is raised from one die;
// see raise_max for what one word costs.  With the maximum over a wave's lanes
// taken by data-parallel primitives, us per step with one word and with eight:
// AugRie 2048^2 with every cell moving 114 -> 107, split step 1024^2 137 -> 125.
constexpr int kCflWords = 8, kCflStride = 32;
struct CflMax {
    unsigned int word[kCflWords * kCflStride];
    __device__ __forceinline__ unsigned bits() const {
        unsigned m = 0u;
#pragma unroll
        for (int i = 0; i < kCflWords; ++i) m = max(m, word[i * kCflStride]);
        return m;
    }
    __device__ __forceinline__ float value() const { return __uint_as_float(bits()); }
    // by the first threads of one workgroup
    __device__ __forceinline__ void clear() {
        if (threadIdx.x < kCflWords) word[threadIdx.x * kCflStride] = 0u;
    }
};

// Device control block of one SWE block: the CFL maxima (three, used in
// turn so that a step can clear the next one without a memset),
// the current dt and simulated time and a per-step dt log.
struct DeviceCtl {
    CflMax smax[3];
    float dt;
    float t;
    int steps;
    int pad[2];
    const unsigned* mlp;  // weight fragments of the learned middle state (solver SOLVER_AUGRIE_MLP)
    unsigned int defer[3];  // edges queued by the deferring sweep, per CFL slot (SOLVER_AUGRIE_DEFER)
    unsigned int busy[3];   // busy record tiles found by the quiet-tile plan of each CFL slot's launch
    // coherent host ring of report_max (kept here rather than passed as a kernel
    // argument, so the launch is an ordinary one)
    unsigned long long* ring;
};

// The CFL maximum of a slot to the host, by one thread: one 64-bit word
// (sequence number above, float bits below) stored at system scope into
// coherent host memory, ctl->ring[seq % kReadbackRing], which the host polls for
// that number.  It needs no event in the stream (an event there costs the
// stream a pause before its next kernel), and the host learns the maximum
// while the stream runs on.
constexpr unsigned kReadbackRing = 4;
__device__ __forceinline__ void report_max(const DeviceCtl* ctl, int slot, unsigned seq) {
    __hip_atomic_store(&ctl->ring[seq % kReadbackRing], ((unsigned long long)seq << 32) | ctl->smax[slot].bits(),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Which CFL-maximum slot a launch reads or accumulates into, and which slot
// it clears for a later step (the last reader of that slot has finished).
struct Slots {
    int use;
    int clear;
};

__device__ __forceinline__ size_t idx(const StateView& v, int x, int y) { return (size_t)x * v.pitch + y; }

// Access to a column that starts at the wave-uniform offset `col` of a field:
// the column's address stays in scalar registers and the load or store adds
// the lane's 32-bit byte offset (lane_bytes).  The empty asm statements keep
// the compiler from forming field + row, or the offset's 64-bit form, once
// per lane outside the column loop: that holds two vector registers for each
// of a sweep's 8 to 15 arrays and costs a vector add per access.  Registers of
// the fused sweeps with 64-bit indices and in this form: HLLE 77 -> 55, f-wave
// 78 -> 56, Hybrid 71 -> 63, AugRie 86 -> 81.
typedef __attribute__((address_space(1))) char GlobalByte;
typedef __attribute__((address_space(1))) float GlobalFloat;
// byte offset of element `row` (non-negative) of a column
__device__ __forceinline__ unsigned lane_bytes(int row) {
    unsigned o = (unsigned)row * 4u;
    asm("" : "+v"(o));
    return o;
}
__device__ __forceinline__ GlobalFloat* col_ptr(const float* f, size_t col, unsigned bytes) {
    GlobalByte* p = (GlobalByte*)const_cast<float*>(f + col);
    asm("" : "+s"(p));
    return (GlobalFloat*)(p + bytes);
}
__device__ __forceinline__ float col_get(const float* f, size_t col, unsigned bytes) { return *col_ptr(f, col, bytes); }
__device__ __forceinline__ void col_set(float* f, size_t col, unsigned bytes, float value) {
    *col_ptr(f, col, bytes) = value;
}

// A store that every lane of the wave executes: lanes that hold nothing to
// store pass kNoStore as their offset, past the column's bound of `pitch`
// elements, and the hardware's range check drops them.  Without a branch
// around it the compiler knows how many stores are in flight and waits for a
// prefetched column's loads only; around a conditional store it has to count
// on the path without it, and so waits for the last column's stores to be
// acknowledged as well, in every column.
constexpr unsigned kNoStore = 0xfffffffcu;
__device__ __forceinline__ void col_put(float* f, size_t col, int pitch, unsigned bytes, float value) {
    __builtin_amdgcn_raw_buffer_store_b32(
        __float_as_uint(value), __builtin_amdgcn_make_buffer_rsrc(f + col, 0, pitch * 4, 0x00020000), bytes, 0, 0);
}

// dt rule of flavour U (SWE_DimensionalSplittingMpi.cpp:448-456)
__device__ __forceinline__ float timestep_from_max(float s, float dx, float dy) {
    if (s > kMinSpeed) {
        float dt = dev::smin(dx / s, dy / s);
        dt *= kCfl;
        return dt;
    }
    return FLT_MAX;
}

// Variant of the sweep, fused and apply kernels (template parameter V): 0 and 1
// are flavour U in IEEE and fast arithmetic, kSplit is flavour S, swe_simple's
// split step (src/blocks/SWE_DimensionalSplitting.cpp:105-210) in IEEE
// arithmetic.  Its y-sweep reads the old state, as flavour U's edges do, so the
// edges, sums and their layout are the same; what differs is
//   the CFL maximum: over the x-edges of all rows, ghost rows included, none of
//                    the y-edges', and dt = 0.4 dx / max without a guard;
//   the update:      Q* = Q - dt/dx (x sums), then h and hv of it - dt/dx (y
//                    sums) -- the y part uses dx too -- without the dry clamp.
constexpr int kSplit = 2;
__host__ __device__ __forceinline__ float split_timestep(float s, float dx) { return kCfl * (dx / s); }

// The maximum over the wave's lanes.  Dpp: by data-parallel-primitive moves
// (within rows of 16 lanes, then across rows), valid in lane 63 and returned as a
// uniform value; for non-negative numbers without NaN.  It takes about a tenth
// of the time of the exchange through LDS.
template <int Ctrl>
__device__ __forceinline__ float dpp_max_step(float v) {
    const int o = __builtin_amdgcn_update_dpp(0, __float_as_int(v), Ctrl, 0xf, 0xf, false);
    return __builtin_fmaxf(v, __int_as_float(o));
}
template <bool Dpp = false>
__device__ __forceinline__ float wave_max(float v) {
    if constexpr (Dpp) {
        v = dpp_max_step<0x111>(v);  // row_shr:1, 2, 4, 8; lanes shifted in read +0
        v = dpp_max_step<0x112>(v);
        v = dpp_max_step<0x114>(v);
        v = dpp_max_step<0x118>(v);
        v = dpp_max_step<0x142>(v);  // row_bcast:15
        v = dpp_max_step<0x143>(v);  // row_bcast:31
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
    } else {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = dev::smax(v, __shfl_xor(v, off, 64));
        return v;
    }
}

// Inclusive sums over the wave's lanes, by data-parallel-primitive moves.
template <int Ctrl, int RowMask>
__device__ __forceinline__ unsigned dpp_add_step(unsigned v) {
    return v + (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, Ctrl, RowMask, 0xf, false);
}
__device__ __forceinline__ unsigned wave_scan(unsigned v) {
    v = dpp_add_step<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = dpp_add_step<0x112, 0xf>(v);
    v = dpp_add_step<0x114, 0xf>(v);
    v = dpp_add_step<0x118, 0xf>(v);
    v = dpp_add_step<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    return dpp_add_step<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// Raise a maximum of the running launch (float bits of a non-negative number)
// to `bits`.  The value only grows while a launch runs, so a wave whose maximum
// does not exceed what it reads leaves it alone, and a stale read costs no more
// than an atomic that changes nothing.  Atomics on one word are served one
// after another, about 12 ns each across the chip's dies, so one atomic per
// wave set a launch's time wherever waves are short.  us per step with an
// atomic per wave and in this form: f-wave 2048^2 in 16-column strips (4352
// waves) 93 -> 62, Hybrid 1500 x 901 90 -> 76, AugRie 2048^2 with every cell
// moving 132 -> 120, 2048^2 islands 43 -> 40, 4096^2 trench 65 -> 49.  (Waves that
// end together all find the old value, hence the several words of a CflMax.)
__device__ __forceinline__ void raise_max(unsigned* m, unsigned bits) {
    if (bits > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(m, bits);
}
__device__ __forceinline__ void raise_max(CflMax& m, unsigned bits) {
    raise_max(&m.word[(blockIdx.x % kCflWords) * kCflStride], bits);
}

// Deferred edges (SOLVER_AUGRIE_DEFER).  An entry is (x, y) of the edge's left
// or lower cell, with kDeferY set in .x for the y-edge (y|y+1); the x-edge is
// (x|x+1).  The batched engine keeps the block index in bits kDeferBlockShift
// and up of .x (blocks < 2^11, x < 2^20).  Each edge is queued once, by the
// lane that owns it: x-edges by the wave whose segment holds x (edge (0|1) by
// the first segment), y-edges by the lane of row y (edge (0|1) by lane 0 of
// the first strip); rows 1..ny only for x-edges.  A deferred edge contributes
// nothing in the sweep: its parts are -0 (x + -0 == x for every x, zeros of
// both signs included, so the sweep stores exactly the other term of each
// two-term sum) and its speed 0.  A second launch adds its parts to the sums
// and its speed to the CFL maximum; IEEE addition is commutative, so every sum
// ends bit for bit as when the edge is solved in the sweep.
constexpr unsigned kDeferY = 0x80000000u;
constexpr int kDeferBlockShift = 20;

__device__ __forceinline__ dev::EdgeOut defer_edge(const dev::EdgeOut& e, bool owns, uint2 entry, uint2* q,
                                                   unsigned* count) {
    const bool d = e.speed < 0.f;
    const unsigned long long m = __ballot(d && owns);
    if (m) {  // uniform over the wave; every lane is active here
        unsigned base = 0;
        if ((threadIdx.x & 63) == 0) base = atomicAdd(count, (unsigned)__popcll(m));
        base = __builtin_amdgcn_readfirstlane(base);
        const unsigned below =
            __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        if (d && owns) q[base + below] = entry;
    }
    return d ? dev::EdgeOut{-0.f, -0.f, -0.f, -0.f, 0.f} : e;
}

// True for the ghost cells that the fused boundary write refreshes after an
// update: corners, and ghost lines of OUTFLOW/WALL sides.
__device__ __forceinline__ bool bc_handles(const StateView& v, const BoundaryInfo& bi, int gx, int gy) {
    auto ow = [](int t) { return t == OUTFLOW || t == WALL; };
    const bool cx = (gx == 0 || gx == v.nx + 1);
    const bool cy = (gy == 0 || gy == v.ny + 1);
    if (cx && cy) return true;
    if (gx == 0) return ow(bi.type[BND_LEFT]);
    if (gx == v.nx + 1) return ow(bi.type[BND_RIGHT]);
    if (gy == 0) return ow(bi.type[BND_BOTTOM]);
    if (gy == v.ny + 1) return ow(bi.type[BND_TOP]);
    return false;
}

// Boundary ghost values of cell (gx, gy) derived from the interior after an
// update: OUTFLOW copies, WALL negates the normal momentum
// (SWE_Block.hh:757-911).  Writes only sides whose type is OUTFLOW/WALL and
// the four corners.
__device__ __forceinline__ void write_boundary_ghosts(const StateView& v, const BoundaryInfo& bi, int x, int y,
                                                      float h, float hu, float hv, float* oh, float* ohu,
                                                      float* ohv) {
    const int nx = v.nx, ny = v.ny;
    if (x == 1) {
        const int t = bi.type[BND_LEFT];
        if (t == OUTFLOW || t == WALL) {
            const size_t g = (size_t)0 * v.pitch + y;
            oh[g] = h;
            ohu[g] = (t == WALL) ? -hu : hu;
            ohv[g] = hv;
        }
    }
    if (x == nx) {
        const int t = bi.type[BND_RIGHT];
        if (t == OUTFLOW || t == WALL) {
            const size_t g = (size_t)(nx + 1) * v.pitch + y;
            oh[g] = h;
            ohu[g] = (t == WALL) ? -hu : hu;
            ohv[g] = hv;
        }
    }
    if (y == 1) {
        const int t = bi.type[BND_BOTTOM];
        if (t == OUTFLOW || t == WALL) {
            const size_t g = (size_t)x * v.pitch + 0;
            oh[g] = h;
            ohu[g] = hu;
            ohv[g] = (t == WALL) ? -hv : hv;
        }
    }
    if (y == ny) {
        const int t = bi.type[BND_TOP];
        if (t == OUTFLOW || t == WALL) {
            const size_t g = (size_t)x * v.pitch + ny + 1;
            oh[g] = h;
            ohu[g] = hu;
            ohv[g] = (t == WALL) ? -hv : hv;
        }
    }
    // corners take the diagonal interior cell whatever the side types
    if (x == 1 && y == 1) {
        oh[0] = h;
        ohu[0] = hu;
        ohv[0] = hv;
    }
    if (x == 1 && y == ny) {
        const size_t g = (size_t)0 * v.pitch + ny + 1;
        oh[g] = h;
        ohu[g] = hu;
        ohv[g] = hv;
    }
    if (x == nx && y == 1) {
        const size_t g = (size_t)(nx + 1) * v.pitch + 0;
        oh[g] = h;
        ohu[g] = hu;
        ohv[g] = hv;
    }
    if (x == nx && y == ny) {
        const size_t g = (size_t)(nx + 1) * v.pitch + ny + 1;
        oh[g] = h;
        ohu[g] = hu;
        ohv[g] = hv;
    }
}

// Flavour-U update of one cell with the dry clamp
// (SWE_DimensionalSplittingMpi.cpp:498-515).
struct Cell {
    float h, hu, hv;
};
__device__ __forceinline__ Cell update_cell(float h, float hu, float hv, float dtdx, float dtdy, float sx, float sy,
                                            float su, float sv) {
    Cell c;
    c.h = h - (dtdx * sx + dtdy * sy);
    c.hu = hu - dtdx * su;
    c.hv = hv - dtdy * sv;
    // a depth below 0 becomes 0, and a cell below the clamp loses its momentum
    const bool thin = c.h < kClampTol;
    c.hu = thin ? 0.f : c.hu;
    c.hv = thin ? 0.f : c.hv;
    c.h = c.h < 0.f ? 0.f : c.h;
    return c;
}

// Variant V's update: flavour S takes dt/dx in both directions and clamps nothing
// (SWE_DimensionalSplitting.cpp:150-168, 196-206).
template <int V>
__device__ __forceinline__ Cell step_cell(float h, float hu, float hv, float dtdx, float dtdy, float sx, float sy,
                                          float su, float sv) {
    if constexpr (V == kSplit)
        return Cell{(h - dtdx * sx) - dtdx * sy, hu - dtdx * su, hv - dtdx * sv};
    else
        return update_cell(h, hu, hv, dtdx, dtdy, sx, sy, su, sv);
}

// One loaded cell: state plus the quantities its edges share.
struct CellQ {
    float h, hu, hv, b, u, v, c, sq, inv, fx, fy;
    __device__ __forceinline__ dev::Side xside() const { return dev::Side{h, hu, b, u, c, sq, inv, fx}; }
    __device__ __forceinline__ dev::Side yside() const { return dev::Side{h, hv, b, v, c, sq, inv, fy}; }
    // the y-side of the cell held by lane + 1 (the cell above), by shuffle
    __device__ __forceinline__ dev::Side yside_from_lane_above() const {
        dev::Side s;
        s.h = __shfl_down(h, 1, 64);
        s.hu = __shfl_down(hv, 1, 64);
        s.b = __shfl_down(b, 1, 64);
        s.u = __shfl_down(v, 1, 64);
        s.c = __shfl_down(c, 1, 64);
        s.sq = __shfl_down(sq, 1, 64);
        s.inv = __shfl_down(inv, 1, 64);
        s.f = __shfl_down(fy, 1, 64);
        return s;
    }
};

template <class A = dev::Ieee>
__device__ __forceinline__ CellQ cell_q(float h, float hu, float hv, float b) {
    CellQ q;
    q.h = h;
    q.hu = hu;
    q.hv = hv;
    q.b = b;
    q.inv = A::rcp(h);
    q.u = hu * q.inv;
    q.v = hv * q.inv;
    q.sq = A::sqrt(h);
    q.c = kSqrtGravity * q.sq;
    q.fx = dev::momentum_flux(h, hu, q.u);
    q.fy = dev::momentum_flux(h, hv, q.v);
    return q;
}

// The two forms of a sweep's tile.  A wave first runs its tile with the short
// divisions and roots of NormalRange and notes any loaded cell outside
// dev::in_normal_range; if there was one, it runs the tile again with the
// compiler's forms and overwrites what it wrote (a tile reads one set of
// buffers and writes another, and reports its maximum only at the end).  The
// general form is cold code after the loop, so it takes no registers from it;
// a choice per column inside the loop spilled (17 registers for AugRie).
// Measured with the short forms and the scalar column addresses (lane_bytes),
// before and after, us per step: 2048^2 islands with every cell moving 163 ->
// 142, 2048^2 islands 48.6 -> 46.0, Hybrid 1500 x 901 117 -> 97; f-wave and HLLE
// are bound by memory and stay.
// body(std::true_type / std::false_type, lane) runs the tile and returns true
// if every cell was in the range.
template <class Ctx, int V, class Body>
__device__ __forceinline__ void run_tile(int lane, const Body& body) {
    if constexpr (V != 1 && Ctx::kNormalForm) {
        if (body(std::true_type(), lane)) return;
        asm volatile("" : "+v"(lane));  // nothing of the general form is computed before
    }
    (void)body(std::false_type(), lane);
}
template <bool N>
using CellMath = std::conditional_t<N, dev::NormalRange, dev::Ieee>;

template <bool N>
__device__ __forceinline__ bool outside_range(const CellQ& q) {
    return N && !dev::in_normal_range(q.h, q.b, q.u, q.v);
}

// Strip sweep.  One wave per (y-tile, x-segment); 4 waves per workgroup.
// dtFixed >= 0 forces dt (the per-call API passes the host's maxTimestep);
// otherwise dt comes from ctl->smax[par].
// The max and store sweeps hold the fused kernel's occupancy target; the
// update sweep of the recompute strategy keeps its natural register use
// (at seven waves it would spill).
template <int S, int MODE, int XS, int V>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == MODE_UPDATE ? 1 : fused_waves_per_simd(S),
                                                                     8))) void sweep_u_kernel(
    StateView v, SumsView sums, float* hn, float* hun, float* hvn, BoundaryInfo bi, DeviceCtl* ctl, Slots sl,
    float dtFixed, int fuseBc, float* dtLog, int logIdx) {
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6));
    const int nyt = (v.ny + kStripRows - 1) / kStripRows;
    const int nxs = (v.nx + XS - 1) / XS;
    if (wave >= nyt * nxs) return;  // uniform per wave
    const dev::SolverCtx<S> solver(S == SOLVER_AUGRIE_MLP ? ctl->mlp : nullptr);
    const int yt = wave % nyt;
    const int xs = wave / nyt;
    const int x0 = 1 + xs * XS;
    const int x1 = min(x0 + XS - 1, v.nx);

    float dtdx = 0.f, dtdy = 0.f, dt = 0.f;
    if (MODE == MODE_UPDATE) {
        dt = dtFixed >= 0.f ? dtFixed : timestep_from_max(ctl->smax[sl.use].value(), v.dx, v.dy);
        dtdx = dt / v.dx;
        dtdy = dt / v.dy;
    }

    auto tile = [&](auto form, int lane) -> bool {
        constexpr bool N = decltype(form)::value;
        using A = CellMath<N>;
        const int y = kStripRows * yt + lane;  // rows y0-1 .. y0+62 with y0 = 62*yt + 1
        const bool rowValid = y <= v.ny + 1;
        const int yc = rowValid ? y : v.ny + 1;
        const bool owned = (lane >= 1) && (lane <= kStripRows) && (y <= v.ny);
        const bool rowInterior = (y >= 1) && (y <= v.ny);
        const bool hEdgeValid = (lane <= kStripRows) && (y <= v.ny);  // edge (y|y+1), y in [0, ny]

        const float* H = v.h;
        const float* HU = v.hu;
        const float* HV = v.hv;
        const float* B = v.b;
        size_t o = (size_t)(x0 - 1) * v.pitch;  // the column's offset, wave-uniform
        unsigned ro = lane_bytes(yc);
        float ch = col_get(H, o, ro), chu = col_get(HU, o, ro), chv = col_get(HV, o, ro), cb = col_get(B, o, ro);
        o += v.pitch;
        float nh = col_get(H, o, ro), nhu = col_get(HU, o, ro), nhv = col_get(HV, o, ro), nb = col_get(B, o, ro);
        // HLLE, f-wave and AugRie load column x+1 one column ahead (a software
        // pipeline: the loads' latency overlaps column x's edges); past x1 + 1
        // the loads stay on column nx + 1 and are not used.
        constexpr bool kAhead = S == SOLVER_HLLE || S == SOLVER_FWAVE || S == SOLVER_AUGRIE;
        float ah = 0.f, ahu = 0.f, ahv = 0.f, ab = 0.f;
        if constexpr (kAhead) {
            o += v.pitch;  // column x0 + 1 <= nx + 1
            ah = col_get(H, o, ro);
            ahu = col_get(HU, o, ro);
            ahv = col_get(HV, o, ro);
            ab = col_get(B, o, ro);
        }

        // In MODE_UPDATE the new buffer must end up a complete state: ghost cells
        // not rewritten by the fused boundary conditions are carried over.  Each
        // ghost row is carried by exactly one lane: row 0 by lane 0 of tile 0,
        // row ny+1 by the tile where it is lane >= 1, other rows by their owner.
        const bool carryRow = owned || (y == 0 && lane == 0) || (y == v.ny + 1 && lane >= 1);
        if (MODE == MODE_UPDATE && x0 == 1 && carryRow && !(fuseBc && bc_handles(v, bi, 0, y))) {
            const size_t g = idx(v, 0, y);
            hn[g] = ch;
            hun[g] = chu;
            hvn[g] = chv;
        }

        // per-cell quantities (velocities, celerity, sqrt h) are computed once
        // when a cell is loaded and reused by its four edges
        CellQ cq = cell_q<A>(ch, chu, chv, cb);
        CellQ nq = cell_q<A>(nh, nhu, nhv, nb);

        bool outside = outside_range<N>(cq) || outside_range<N>(nq);

        // halo vertical edge (x0-1 | x0)
        const dev::EdgeOut e = solver.template solve<A>(cq.xside(), nq.xside());
        float carryH = e.hR, carryHu = e.huR;
        const bool xCounts = V == kSplit ? rowValid : rowInterior;
        float smaxv = !xCounts ? 0.f : V == kSplit ? dev::smax(0.f, e.speed) : e.speed;

        for (int x = x0; x <= x1; ++x) {
            ch = nh;
            chu = nhu;
            chv = nhv;
            cb = nb;
            cq = nq;
            if constexpr (kAhead) {
                nh = ah;
                nhu = ahu;
                nhv = ahv;
                nb = ab;
                if (x + 2 <= v.nx + 1) o += v.pitch;  // column x+2, else stay on nx+1
                ro = lane_bytes(yc);
                ah = col_get(H, o, ro);
                ahu = col_get(HU, o, ro);
                ahv = col_get(HV, o, ro);
                ab = col_get(B, o, ro);
            } else {
                o += v.pitch;  // column x+1 (<= nx+1)
                ro = lane_bytes(yc);
                nh = col_get(H, o, ro);
                nhu = col_get(HU, o, ro);
                nhv = col_get(HV, o, ro);
                nb = col_get(B, o, ro);
            }
            nq = cell_q<A>(nh, nhu, nhv, nb);
            outside = outside || outside_range<N>(nq);

            // vertical edge (x | x+1)
            const dev::EdgeOut ev = solver.template solve<A>(cq.xside(), nq.xside());
            if (xCounts) smaxv = dev::smax(smaxv, ev.speed);

            // horizontal edge (y | y+1): upper cell from lane+1
            const dev::EdgeOut eh = solver.template solve<A>(cq.yside(), cq.yside_from_lane_above());
            if (V != kSplit && hEdgeValid) smaxv = dev::smax(smaxv, eh.speed);
            // up-going part of edge (y-1 | y) from lane-1
            const float aH = __shfl_up(eh.hR, 1, 64);
            const float aHv = __shfl_up(eh.huR, 1, 64);

            const float sx = carryH + ev.hL;
            const float su = carryHu + ev.huL;
            const float sy = aH + eh.hL;
            const float sv = aHv + eh.huL;
            carryH = ev.hR;
            carryHu = ev.huR;

            const size_t c = (size_t)x * v.pitch;
            if (MODE == MODE_STORE && owned) {
                const unsigned ry = lane_bytes(y);
                col_set(sums.sx, c, ry, sx);
                col_set(sums.sy, c, ry, sy);
                col_set(sums.su, c, ry, su);
                col_set(sums.sv, c, ry, sv);
            }
            if (MODE == MODE_UPDATE) {
                const unsigned ry = lane_bytes(y);
                if (owned) {
                    const Cell nc = update_cell(ch, chu, chv, dtdx, dtdy, sx, sy, su, sv);
                    col_set(hn, c, ry, nc.h);
                    col_set(hun, c, ry, nc.hu);
                    col_set(hvn, c, ry, nc.hv);
                    if (fuseBc) write_boundary_ghosts(v, bi, x, y, nc.h, nc.hu, nc.hv, hn, hun, hvn);
                } else if (carryRow && (y == 0 || y == v.ny + 1) && !(fuseBc && bc_handles(v, bi, x, y))) {
                    col_set(hn, c, ry, ch);  // carry ghost rows into the new buffer
                    col_set(hun, c, ry, chu);
                    col_set(hvn, c, ry, chv);
                }
            }
        }
        if (MODE == MODE_UPDATE && x1 == v.nx && carryRow && !(fuseBc && bc_handles(v, bi, v.nx + 1, y))) {
            const size_t g = idx(v, v.nx + 1, y);
            hn[g] = nh;
            hun[g] = nhu;
            hvn[g] = nhv;
        }

        if (N && __any(outside)) return false;
        if (MODE != MODE_UPDATE) {
            smaxv = wave_max<N>(smaxv);
            if (lane == 0) raise_max(ctl->smax[sl.use], __float_as_uint(smaxv));
        }
        return true;
    };
    run_tile<dev::SolverCtx<S>, V>(threadIdx.x & 63, tile);

    if (MODE == MODE_UPDATE) {
        if (blockIdx.x == 0) ctl->smax[sl.clear].clear();  // a later step's maximum starts from zero
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            if (dtFixed < 0.f) {
                ctl->dt = dt;
                ctl->t += dt;
                ctl->steps += 1;
                if (dtLog) dtLog[logIdx] = dt;
            }
        }
    }
}

// Apply stored net-update sums in place (second half of the store strategy).
template <int XS, int V>
__global__ __launch_bounds__(256) void apply_u_kernel(StateView v, SumsView sums, BoundaryInfo bi, DeviceCtl* ctl,
                                                       Slots sl, float dtFixed, int fuseBc, float* dtLog,
                                                       int logIdx) {
    const int y = blockIdx.x * 64 + (threadIdx.x & 63) + 1;
    const int xseg = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int x0 = 1 + xseg * XS;
    const float dt = dtFixed >= 0.f ? dtFixed : timestep_from_max(ctl->smax[sl.use].value(), v.dx, v.dy);
    const float dtdx = dt / v.dx;
    const float dtdy = dt / v.dy;
    if (y <= v.ny && x0 <= v.nx) {
        const int x1 = min(x0 + XS - 1, v.nx);
        for (int x = x0; x <= x1; ++x) {
            const size_t c = idx(v, x, y);
            const Cell nc = update_cell(v.h[c], v.hu[c], v.hv[c], dtdx, dtdy, sums.sx[c], sums.sy[c], sums.su[c],
                                        sums.sv[c]);
            v.h[c] = nc.h;
            v.hu[c] = nc.hu;
            v.hv[c] = nc.hv;
            if (fuseBc) write_boundary_ghosts(v, bi, x, y, nc.h, nc.hu, nc.hv, v.h, v.hu, v.hv);
        }
    }
    if (blockIdx.x == 0 && blockIdx.y == 0) ctl->smax[sl.clear].clear();
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (dtFixed < 0.f) {
            ctl->dt = dt;
            ctl->t += dt;
            ctl->steps += 1;
            if (dtLog) dtLog[logIdx] = dt;
        }
    }
}

}  // namespace swe
