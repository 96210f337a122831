// Pit filling: PitFillingAlgorithm<T>::execute, PitFillingAlgorithm.h:88-98,
// parity target performPitFilling, PitFillingAlgorithmCPUOpenMP.h:68-242.
//
// What the reference computes.  After quantising to mm (:84-106) it floods
// from the seeds (non-nodata edge cells and cells at 0) through buckets of
// 1/1000 m in increasing order (:162-237).  A popped cell c expands its
// unprocessed 8-neighbours n to max(z_n, spill_c); every cell is pushed once,
// into bucket toIndex(v) of its value v, and when popped it expands only if
// toElev(toIndex(v)) == v (:178-181).  Values that fail that round trip
// ("dead" values, e.g. 0.251 m) never expand, so with P the result
//   P(n) = max(Z(n), min { P(c) : c an 8-neighbour, reached, live(P(c)) }),
// seeds fixed at Z, unreached cells keep Z.
//
// How it is computed here: two bounds, no priority queue.  A cell raised
// above its Z takes a neighbour's relayed value, which is live, so only
// cells whose own Z is dead can be dead: with m(n) the least value relayed to
// such a cell, it is blocked (P(n) = Z(n), relays nothing) when m(n) <= Z(n)
// and relays m(n) like any other cell when m(n) > Z(n).  For a fixed choice
// of the blocked cells the result is the greatest fixed point of
//   W(n) = max(Z(n), min relay(c)),
// reached from +inf by monotone relaxation in any order.  Blocking more
// cells only raises it, so it brackets P:
//   upper bound U: every dead cell not proven to relay is blocked;
//   lower bound L: every dead cell not proven blocked relays.
// A dead cell with m_U <= Z is blocked for certain (P <= U), one with
// m_L > Z relays for certain (P >= L).  Stages alternate:
//   stage 0 (U): every dead cell blocked, from +inf;
//   odd stages (L): from U, the dead cells with m_U > Z relay too;
//   even stages (U): from U, those of them with m_L > Z relay for good.
// Each starts from the last U, a valid upper start, so after stage 0 only the
// cells behind a dead cell are touched (0.4 % of a 4096^2 realization).
// When an L stage ends with every relaying dead cell above its Z the choice is
// consistent and L is P.  While one is not, the U stage proves at least the
// lowest of them, so the stages end.  A 4096^2 realization takes 3 L stages.
//
// Execution: one persistent launch without grid barriers.  Every 64 x 64
// tile belongs to the workgroup that takes it in stage 0 (a workgroup takes
// the next when done with one), which holds the tile it worked on last in LDS;
// with as many workgroups as tiles none is ever loaded twice.  Tiles talk
// through an exchange buffer that holds each tile's four border rows and
// columns: a workgroup that lowers a border cell stores its side there and
// marks the rows this unsettles in the neighbour's flag word, if any can
// change; the neighbour's owner finds the mark when it next polls, reloads
// the ring and solves those rows.  A stage is over when no flag is up and no
// tile is at work (see pf_publish).
//
// What bounds it: at 4096^2 the row steps' issue (four waves a SIMD), below
// 1024 tiles the chain of dependent visits (a visit's solve plus some 5 us
// from a published side to the neighbour's reload).  The form it replaced
// (pitfill_rounds.hip) ran 60 barrier-separated passes of fill and
// certification, each ending with its slowest tile.  Times of the stage, the
// benchmark's Gaussian realizations, that form / this one: 128 x 96 0.19 /
// 0.08 ms, 1000 x 777 2.04 / 0.44, 2048^2 2.28 / 0.57, 4096^2 4.09 / 1.11,
// 8192^2 7.39 / 2.69.
//
// Every comparison is on floats; the only arithmetic is the quantisation and
// the round-trip test, both evaluated exactly as the reference does.
#include <vector>

#include "tiles.hpp"

namespace cageo {

namespace {

constexpr float PF_INF = __builtin_huge_valf();

struct PfShared {
    float rel[HALO_W * HALO_W];   // relays of the tile and its ring, +inf: none
    uint32_t rowdirty[TILE];      // strip edge rows marked by the neighbouring strips
    unsigned long long can[TILE_THREADS / 64];  // ring cells of sides N, S, W, E to be lowered
    uint32_t bits;                // PF_BIT_* of the visit
    int cmd;                      // wave 0's poll: tile to visit, or PF_DONE / PF_ABANDON
    uint32_t rows_lo, rows_hi;    // rows of that tile to solve
};

// Z of a thread's 16 cells (row k of its strip): a vector, so that the
// sweeps' read of row k (the same k across the wave) is an indexed register
// move, where an array would live in scratch.
typedef float ZRow __attribute__((ext_vector_type(STRIP)));

constexpr int PF_DONE = -1;     // the stage is over
constexpr int PF_ABANDON = -2;  // the launch is being abandoned
constexpr uint32_t PF_OVER_ABANDON = 0xffffffffu;

// Words of a group's line of the stage counters.
constexpr int PF_ASKED = 0;  // visits asked for: flags raised, and the first visits of each workgroup
constexpr int PF_ENDED = 1;  // visits ended
constexpr int PF_LOW = 2;    // undecided cells at their Z

// PfShared::bits: sides 0-3 hold a cell lowered in the visit; the ring's
// corners 0-3 (NW, NE, SW, SE) can be lowered; undecided cells are left.
constexpr uint32_t PF_BIT_SIDE = 1u, PF_BIT_CORNER = 1u << 4, PF_BIT_DEAD = 1u << 8;

// Per-tile word of its owner.
constexpr uint32_t PF_INFO_DEAD = 1;  // holds undecided dead cells
constexpr uint32_t PF_INFO_LPUB = 2;  // its lower-bound sides differ from the upper bound's
constexpr uint32_t PF_INFO_INF = 4;   // written back with cells still at +inf
constexpr uint32_t PF_INFO_LOW = 8;   // its lower bound of this stage is in R.low

constexpr int PF_SIDE = 64;           // cells of a side in the exchange buffer
constexpr int PF_SIDES = 4 * PF_SIDE; // north, south rows, west, east columns
// Planes of the exchange buffer: relays of the upper and the lower bound, and
// Z (negated for a dead cell, +inf for one that never relays; 0 until the
// tile's first visit).
enum : int { PF_UPPER = 0, PF_LOWER = 1, PF_FLOOR = 2, PF_PLANES = 3 };

__device__ inline float min8(const float* s, int i) {
    const float a = fminf(fminf(s[i - HALO_W - 1], s[i - HALO_W]), fminf(s[i - HALO_W + 1], s[i - 1]));
    const float b = fminf(fminf(s[i + 1], s[i + HALO_W - 1]), fminf(s[i + HALO_W], s[i + HALO_W + 1]));
    return fminf(a, b);
}

__device__ inline uint32_t ld(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Waits until this wave's stores and atomics are performed: an agent-scope
// store issued before is then visible to every workgroup.
__device__ inline void wait_stores() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
}

// One raster of a launch.
struct PfRaster {
    const float* zq;
    float* w;
    float* low;  // scratch of the raster's size: lower bounds of tiles that left LDS
    int W, H, ntx, nty;
    float nodata;
    const uint32_t* __restrict__ scal;  // min/max/bad of the quantized raster
    uint32_t* status;      // the raster's sticky status word
};

// A launch over one raster (`one`, rs null) or over the rasters of a table,
// whose 64x64 blocks are numbered globally (bmap).
struct PfArgs {
    PfRaster one;
    const PfRaster* __restrict__ rs;
    const int2* __restrict__ bmap;  // per block: (raster, block within it)
    uint32_t total;                 // blocks
    uint32_t most;                  // blocks a workgroup takes at most
    int* own;                       // most x workgroups: the blocks each took
    unsigned long long* flags;      // 2 stage parities x total: rows to solve
    float* xb;       // PF_PLANES x total x PF_SIDES: the tiles' sides
    uint2* masks;    // total x 256: a thread's obst | dead << 16, low (see PfTile)
    uint32_t* info;  // total: PF_INFO_*
    uint32_t* ctrl;  // control block (CTL_*)
    GridBar gb;      // status, abort words and wait bound (no barrier is used)
};

// The counters of `group` in `stage`.
__device__ inline uint32_t* pf_counts(const PfArgs& a, uint32_t stage, uint32_t group) {
    return a.ctrl + CTL_PF_COUNTS + (stage & 3u) * CTL_PF_STAGE + group * CTL_PF_LINE;
}
__device__ inline uint32_t* pf_own_counts(const PfArgs& a, uint32_t stage) {
    return pf_counts(a, stage, blockIdx.x % CTL_PF_GROUPS);
}
// Block j of the workgroup's own.
__device__ inline uint32_t pf_own(const PfArgs& a, uint32_t j) {
    return (uint32_t)a.own[(size_t)j * gridDim.x + blockIdx.x];
}
// Sum of counter `word` over the groups (every lane of the calling wave).
__device__ inline uint32_t pf_sum(const PfArgs& a, uint32_t stage, int word) {
    static_assert(CTL_PF_GROUPS == 64, "a lane a group");
    int v = (int)ld(pf_counts(a, stage, threadIdx.x & 63) + word), zero = 0;
    auto add = [](int& s, int&, int p, int) { s += p; };
    CAGEO_SCAN_UP(dpp_i, v, zero, 0, 0, add);
    return (uint32_t)lane_read(v, 63);
}

// The raster of global block g, g's number within it, and the raster's
// minimum and domain flag (`mn1`, `ok1` for a one-raster launch).
struct PfBlock {
    PfRaster R;
    int lb, gbase;
    float mn;
    bool ok;
};

// Domain of the reference's arithmetic: non-negative elevations and a bucket
// array fl(fl(max-min)*1000)+1 that float arithmetic indexes exactly (beyond
// 2^24 the reference reads past it).  Sets the raster's minimum.
// The scalars were written by an earlier launch and are read-only here, so
// plain (cacheable) loads are exact.
__device__ inline bool pf_raster_ok(const PfRaster& R, float& mn) {
    const uint32_t bad = R.scal[SC_BAD];
    mn = ordered_to_float(R.scal[SC_MIN]);
    const float mx = ordered_to_float(R.scal[SC_MAX]);
    const float span = (mx - mn) * 1000.0f;
    return !bad && span < 16777216.0f;
}

template <bool MULTI>
__device__ inline PfBlock pf_block(const PfArgs& a, uint32_t g, float mn1, bool ok1) {
    PfBlock b;
    g = __builtin_amdgcn_readfirstlane(g);
    if constexpr (!MULTI) {
        b.R = a.one;
        b.lb = (int)g;
        b.mn = mn1;
        b.ok = ok1;
    } else {
        const int2 m = a.bmap[g];
        const int r = __builtin_amdgcn_readfirstlane(m.x);
        b.lb = __builtin_amdgcn_readfirstlane(m.y);
        b.R = a.rs[r];
        b.ok = pf_raster_ok(b.R, b.mn);
    }
    b.gbase = (int)g - b.lb;
    return b;
}

// The tile a workgroup holds in LDS and each thread's part of it: masks over
// its strip's 16 cells (bit k = row k).
struct PfTile {
    int tile = -1;
    bool lower = false;  // LDS holds the lower bound
    ZRow zr;             // Z
    uint32_t obst = 0;   // relays nothing in the upper bound: nodata, outside the
                         // raster, dead seeds, dead cells not proven to relay
    uint32_t dead = 0;   // of those, the dead cells not proven blocked either
    uint32_t low = 0;    // of those, the ones at their Z in the lower bound
    uint32_t chg = 0;    // cells not yet written back
};

// Row solves of a tile whose relays are in LDS, over the rows `rd` of the
// strip first (see strip_rows) and then every row a change reaches.  Cells
// in `obst` relay nothing; `lowered` collects the cells whose value dropped.
//
// Row step (all 64 columns at once): a cell is the map
// v -> max(Z, min(c, v)), c = min(its value, the relays above and below), a
// clamp to [Z, max(Z, c)]; a seed's value is its Z and an obstacle's Z counts
// as +inf, so both are constant maps.  The fixed point of the row,
// W(x) = max(Z, min(c, W(x-1), W(x+1))), is min(L(x), R(x)) with L, R the
// map chains from the left and right halo cells.  About 150 instructions,
// bound by the latency of the two scans; a row whose cells all sit at their
// Z (or relay nothing) cannot change and is skipped after one read.
__device__ inline void fill_sweeps(PfShared& S, uint32_t rd, const ZRow& zr, uint32_t obst,
                                   uint32_t& lowered) {
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ClampCarry cc;
    clamp_carry_init(cc);
    for (int sweep = 0;; ++sweep) {
        int changed = 0;
        const bool upward = sweep_upward(S.rowdirty, rd, strip, sweep);
        for (int kk = 0; kk < STRIP; ++kk) {
            const int k = upward ? (STRIP - 1 - kk) : kk;
            const int ly = strip * STRIP + k;
            if (!row_due(S.rowdirty, rd, k, ly)) continue;
            const int li = (ly + 1) * HALO_W + lx + 1;
            // the step's reads at once: the cell, its neighbours in the rows
            // above and below, and the row's two halo cells (one address for
            // the whole wave)
            const float c = S.rel[li];
            const float a0 = S.rel[li - HALO_W - 1], a1 = S.rel[li - HALO_W], a2 = S.rel[li - HALO_W + 1];
            const float b0 = S.rel[li + HALO_W - 1], b1 = S.rel[li + HALO_W], b2 = S.rel[li + HALO_W + 1];
            const float hlv = __int_as_float(__builtin_amdgcn_readfirstlane(
                __float_as_int(S.rel[(ly + 1) * HALO_W])));
            const float hrv = __int_as_float(__builtin_amdgcn_readfirstlane(
                __float_as_int(S.rel[(ly + 1) * HALO_W + HALO_W - 1])));
            // Z, +inf for an obstacle
            const float z = fmaxf(zr[k], __int_as_float(__builtin_amdgcn_sbfe((int)obst, k, 1) & 0x7f800000));
            if (__ballot(c > z) == 0) continue;
            const float m6 = fminf(fminf(fminf(a0, a1), fminf(a2, b0)), fminf(b1, b2));
            // what a row holds is no fixed point while some cell is above what its
            // eight neighbours allow it (the end lanes keep the halo cells; the
            // moves are outside any branch, where a lane switched off could not
            // be read)
            const float m2 = fminf(dpp_f<DPP_WAVE_SHR1>(hlv, c), dpp_f<DPP_WAVE_SHL1>(hrv, c));
            if (__ballot(fmaxf(z, fminf(m6, m2)) < c) == 0) continue;
            float llo = z, lhi = fmaxf(z, fminf(c, m6));
            float rlo = llo, rhi = lhi;
            scan_clamp_up(llo, lhi, cc);
            scan_clamp_down(rlo, rhi, cc);
            const float nw = fminf(clamp3(hlv, llo, lhi), clamp3(hrv, rlo, rhi));
            const bool ch = nw < c;
            if (ch) {
                S.rel[li] = nw;
                lowered |= 1u << k;
            }
            if (__ballot(ch)) {
                changed = 1;
                row_mark(S.rowdirty, rd, k, ly);
            }
        }
        if (!__syncthreads_or(changed)) break;
    }
}

// Sides of tile g in a plane of the exchange buffer.
__device__ inline float* pf_sides(const PfArgs& a, int plane, uint32_t g) {
    return a.xb + ((size_t)plane * a.total + g) * PF_SIDES;
}
__device__ inline float ld_side(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_side(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Cell p of a tile's side 0..3 in the LDS tile; `out` cells outside it (1: the
// ring's cell beside it).
__device__ inline int side_cell(int side, int p, int out) {
    return side == 0 ? (1 - out) * HALO_W + p + 1 : side == 1 ? (TILE + out) * HALO_W + p + 1
         : side == 2 ? (p + 1) * HALO_W + 1 - out : (p + 1) * HALO_W + TILE + out;
}
// The ring's corner 0..3 (NW, NE, SW, SE).
__device__ inline int corner_cell(int corner) {
    return (corner < 2 ? 0 : HALO_W - 1) * HALO_W + ((corner & 1) ? HALO_W - 1 : 0);
}

// Loads the ring of the tile: wave 0 the row above it, wave 1 the row below,
// waves 2 and 3 the columns beside it, lane 0 of each wave one corner.
// `floor` and `cfloor` get the least value this thread's cell and corner can
// take in this stage, +inf for one that cannot change.  Returns whether
// they hold a relay.
__device__ inline bool load_ring(PfShared& S, const PfArgs& a, const PfBlock& b, uint32_t stage,
                                 bool lower, float& floor, float& cfloor) {
    const int p = threadIdx.x & 63, side = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tx = b.lb % b.R.ntx, ty = b.lb / b.R.ntx;
    // the neighbour across this wave's side, and at its corner: there the cell
    // lies in the neighbour's south (1) or north (0) row
    const int dx = side < 2 ? 0 : (side == 2 ? -1 : 1), dy = side == 0 ? -1 : side == 1 ? 1 : 0;
    const int cx = (side & 1) ? 1 : -1, cy = side < 2 ? -1 : 1;
    const bool in = tx + dx >= 0 && tx + dx < b.R.ntx && ty + dy >= 0 && ty + dy < b.R.nty;
    const bool cin = tx + cx >= 0 && tx + cx < b.R.ntx && ty + cy >= 0 && ty + cy < b.R.nty;
    const int plane = lower ? PF_LOWER : PF_UPPER;
    float v = PF_INF, cv = PF_INF;
    floor = cfloor = PF_INF;
    if (in) {
        const uint32_t g = (uint32_t)(b.gbase + (ty + dy) * b.R.ntx + tx + dx);
        const int o = (side ^ 1) * PF_SIDE + p;
        v = ld_side(pf_sides(a, plane, g) + o);
        floor = ld_side(pf_sides(a, PF_FLOOR, g) + o);
    }
    if (cin && p == 0) {
        const uint32_t g = (uint32_t)(b.gbase + (ty + cy) * b.R.ntx + tx + cx);
        const int o = (side < 2 ? PF_SIDE : 0) + ((side & 1) ? 0 : PF_SIDE - 1);
        cv = ld_side(pf_sides(a, plane, g) + o);
        cfloor = ld_side(pf_sides(a, PF_FLOOR, g) + o);
    }
    S.rel[side_cell(side, p, 1)] = v;
    if (p == 0) S.rel[corner_cell(side)] = cv;
    // in stage 0 no dead cell relays
    floor = floor < 0.0f && stage == 0 ? PF_INF : fabsf(floor);
    cfloor = cfloor < 0.0f && stage == 0 ? PF_INF : fabsf(cfloor);
    return v < PF_INF || cv < PF_INF;
}

// What a visit starts with (before a barrier).
__device__ inline void visit_reset(PfShared& S) {
    if (threadIdx.x < TILE) S.rowdirty[threadIdx.x] = 0u;
    if (threadIdx.x == 0) S.bits = 0u;
}

// First load of tile `t`: cells from Z alone (PitFillingAlgorithmCPUOpenMP.h:
// 121-144 seeds), +inf where nothing has reached them yet.  The cells that
// relay nothing get their final value, Z, in the output at once.  Returns the
// thread's cells that relay already (seeds).
__device__ inline uint32_t load_first(PfShared& S, PfTile& T, const PfBlock& b) {
    const PfRaster& R = b.R;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = (b.lb % R.ntx) * TILE + lx, y0 = (b.lb / R.ntx) * TILE + strip * STRIP;
    // every load issued before one is used (a cell outside loads cell 0), and
    // the stores after them all: a store between would have to be waited for
    float zv[STRIP];
#pragma unroll
    for (int k = 0; k < STRIP; ++k)
        zv[k] = R.zq[x < R.W && y0 + k < R.H ? (size_t)(y0 + k) * R.W + x : 0];
    uint32_t obst = 0, dead = 0, seeds = 0, inside = 0;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const int y = y0 + k;
        const float z = zv[k];
        const bool in = x < R.W && y < R.H;
        const bool live = in && z != R.nodata && pf_live(z, b.mn);
        const bool seed = x == 0 || y == 0 || x == R.W - 1 || y == R.H - 1 || z == 0.0f;
        if (in) inside |= 1u << k;
        if (!live) obst |= 1u << k;
        if (live && seed) seeds |= 1u << k;
        if (in && !live && !seed && z != R.nodata) dead |= 1u << k;
        S.rel[(strip * STRIP + k + 1) * HALO_W + lx + 1] = live && seed ? z : PF_INF;
        T.zr[k] = z;
    }
#pragma unroll
    for (int k = 0; k < STRIP; ++k)
        if (((inside & obst) >> k) & 1u) R.w[(size_t)(y0 + k) * R.W + x] = zv[k];
    T.obst = obst;
    T.dead = dead;
    T.low = 0;
    T.chg = inside & ~obst;
    return seeds;
}

// Stores the floors of the tile's sides, held by the lanes of its border.
__device__ inline void put_floors(const PfTile& T, const PfArgs& a) {
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* s = pf_sides(a, PF_FLOOR, (uint32_t)T.tile);
    auto floor = [&](int k) {
        return ((T.dead >> k) & 1u) ? -T.zr[k] : ((T.obst >> k) & 1u) ? PF_INF : T.zr[k];
    };
    if (strip == 0) st_side(s + lx, floor(0));
    if (strip == TILE / STRIP - 1) st_side(s + PF_SIDE + lx, floor(STRIP - 1));
    if (lx == 0 || lx == TILE - 1) {
#pragma unroll
        for (int k = 0; k < STRIP; ++k)
            st_side(s + (lx == 0 ? 2 : 3) * PF_SIDE + strip * STRIP + k, floor(k));
    }
}

// Loads the upper bound (or with `low` the lower bound) of tile `t` again, its
// ring apart.
__device__ inline void load_again(PfShared& S, PfTile& T, const PfArgs& a, const PfBlock& b,
                                  uint32_t t, bool low) {
    const PfRaster& R = b.R;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = (b.lb % R.ntx) * TILE + lx, y0 = (b.lb / R.ntx) * TILE + strip * STRIP;
    float zv[STRIP], wv[STRIP];
    const float* src = low ? R.low : R.w;
    const uint2 m = a.masks[(size_t)t * TILE_THREADS + threadIdx.x];
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const size_t gi = x < R.W && y0 + k < R.H ? (size_t)(y0 + k) * R.W + x : 0;
        zv[k] = R.zq[gi];
        wv[k] = src[gi];  // (cells outside are in obst)
    }
    T.obst = m.x & 0xffffu;
    T.dead = m.x >> 16;
    T.low = m.y;
    T.chg = 0;
    T.lower = low;
    T.tile = (int)t;
    const uint32_t none = low ? T.obst & ~T.dead : T.obst;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        S.rel[(strip * STRIP + k + 1) * HALO_W + lx + 1] = (none >> k) & 1u ? PF_INF : wv[k];
        T.zr[k] = zv[k];
    }
}

// Writes the thread's cells of `T.chg` back, with `last` a cell never reached
// as its Z.  Returns whether one of them was left at +inf.
__device__ inline bool write_cells(PfShared& S, PfTile& T, const PfBlock& b, bool last) {
    const PfRaster& R = b.R;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = (b.lb % R.ntx) * TILE + lx, y0 = (b.lb / R.ntx) * TILE + strip * STRIP;
    bool inf = false;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        float v = S.rel[(strip * STRIP + k + 1) * HALO_W + lx + 1];
        const bool none = !(v < PF_INF);
        // (a cell written back at +inf before is not in chg any more)
        if (!((T.chg >> k) & 1u) && !(last && none && !((T.obst >> k) & 1u))) continue;
        inf = inf || none;
        if (last && none) v = T.zr[k];
        R.w[(size_t)(y0 + k) * R.W + x] = v;
    }
    T.chg = 0;
    return inf;
}

// Writes the lower bound of the thread's cells out (true: it is there).
__device__ inline bool write_low(const PfShared& S, const PfTile& T, const PfBlock& b) {
    const PfRaster& R = b.R;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = (b.lb % R.ntx) * TILE + lx, y0 = (b.lb / R.ntx) * TILE + strip * STRIP;
#pragma unroll
    for (int k = 0; k < STRIP; ++k)
        if (x < R.W && y0 + k < R.H)
            R.low[(size_t)(y0 + k) * R.W + x] = S.rel[(strip * STRIP + k + 1) * HALO_W + lx + 1];
    return true;
}

// Writes the bound held in LDS back, before LDS takes another tile or goes on
// as the lower bound.  In a U stage (`lower` false) a lower bound is done with.
template <bool MULTI>
__device__ inline void flush_tile(PfShared& S, PfTile& T, const PfArgs& a, bool lower, float mn1,
                                  bool ok1) {
    if (T.tile < 0) return;
    a.masks[(size_t)T.tile * TILE_THREADS + threadIdx.x] = make_uint2(T.obst | (T.dead << 16), T.low);
    const PfBlock b = pf_block<MULTI>(a, (uint32_t)T.tile, mn1, ok1);
    bool mark = false;
    if (!T.lower) mark = write_cells(S, T, b, false);
    else if (lower) mark = write_low(S, T, b);
    if (__syncthreads_or(mark) && threadIdx.x == 0)
        a.info[T.tile] |= T.lower ? PF_INFO_LOW : PF_INFO_INF;
}

// Ends a visit: publishes the sides that hold a lowered cell and raises the
// neighbours' flags.  In a U stage both planes get the sides, so that an L
// stage starts with the two alike; `all_lower` rewrites every side of the
// lower plane (a U stage's first visit to a tile the L stage before changed).
//
// A stage is over when as many visits ended as were asked for.  A visit that
// raises flags first counts one for each neighbour as asked for, before a flag
// can be seen, and counts the flags that were up already as ended with its
// own end, after the last is raised; so while work is left, fewer are ended
// than asked for.  Both only grow, so reading the ended counts of all groups
// before the asked ones and finding the sums equal proves the stage over.
__device__ inline void pf_publish(PfShared& S, const PfTile& T, const PfArgs& a, const PfBlock& b,
                                  uint32_t stage, uint32_t lowered, float floor, float cfloor,
                                  uint32_t share, bool all_lower) {
    const bool lower = stage & 1;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // sides with a cell lowered in this visit
    uint32_t bits = 0;
    if (__ballot(lx == 0 && lowered)) bits |= PF_BIT_SIDE << 2;
    if (__ballot(lx == TILE - 1 && lowered)) bits |= PF_BIT_SIDE << 3;
    if (strip == 0 && __ballot(lowered & 1u)) bits |= PF_BIT_SIDE;
    if (strip == TILE / STRIP - 1 && __ballot(lowered >> (STRIP - 1))) bits |= PF_BIT_SIDE << 1;
    if (__ballot(T.dead != 0u)) bits |= PF_BIT_DEAD;
    // ring cells of this wave's side, and its corner, that the tile's border
    // can lower: higher than the border cells beside them and than their own
    // least value
    {
        const int c = side_cell(strip, lx, 0), step = strip < 2 ? 1 : HALO_W;
        float m = S.rel[c];
        if (lx > 0) m = fminf(m, S.rel[c - step]);
        if (lx < PF_SIDE - 1) m = fminf(m, S.rel[c + step]);
        const unsigned long long can = __ballot(S.rel[side_cell(strip, lx, 1)] > fmaxf(floor, m));
        const float cm = S.rel[side_cell(strip < 2 ? 0 : 1, (strip & 1) ? PF_SIDE - 1 : 0, 0)];
        const bool cc = lx == 0 && S.rel[corner_cell(strip)] > fmaxf(cfloor, cm);
        if (__ballot(cc)) bits |= PF_BIT_CORNER << strip;
        if (lx == 0) {
            S.can[strip] = can;
            if (bits) atomicOr(&S.bits, bits);
        }
    }
    __syncthreads();
    const uint32_t all = (uint32_t)__builtin_amdgcn_readfirstlane((int)S.bits);
    const bool border = (all & 0xfu) != 0u;
    uint32_t* counts = pf_own_counts(a, stage);
    // neighbours to call, in TDX / TDY order (lanes 0-7 of wave 0): across a
    // side for the rows of its cells that can be lowered, at a corner for one
    bool call = false;
    unsigned long long rows = 0;
    if (threadIdx.x < 8 && border) {
        // N, NE, E, SE, S, SW, W, NW: side or 4 + corner, a nibble each
        const int w = (int)((0x42617350u >> (4 * lx)) & 7u);
        if (w < 4) {
            rows = S.can[w];
            call = rows != 0ull;
            if (w == 0) rows = 1ull << (TILE - 1);
            if (w == 1) rows = 1ull;
        } else {
            call = (all >> w) & 1u;
            rows = w < 6 ? 1ull << (TILE - 1) : 1ull;
        }
    }
    const uint32_t asked = (uint32_t)__popcll(__ballot(call));  // (wave 0)
    if (border || all_lower) {
        const float v = S.rel[side_cell(strip, lx, 0)];
        const size_t o = (size_t)strip * PF_SIDE + lx;
        const bool mine = (all >> strip) & 1u;
        if (!lower && mine) st_side(pf_sides(a, PF_UPPER, (uint32_t)T.tile) + o, v);
        if (mine || all_lower) st_side(pf_sides(a, PF_LOWER, (uint32_t)T.tile) + o, v);
    }
    if (threadIdx.x == 0 && asked) atomicAdd(&counts[PF_ASKED], asked);
    wait_stores();
    __syncthreads();
    if (threadIdx.x < 64) {
        bool up = false;
        if (call) {
            const int nx = b.lb % b.R.ntx + TDX[lx], ny = b.lb / b.R.ntx + TDY[lx];
            unsigned long long* f = a.flags + (size_t)(stage & 1u) * a.total + b.gbase +
                                    ny * b.R.ntx + nx;
            up = __hip_atomic_fetch_or(f, rows, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0ull;
        }
        const uint32_t newly = (uint32_t)__popcll(__ballot(up));
        if (threadIdx.x == 0) {
            uint32_t inf = a.info[T.tile] & ~PF_INFO_DEAD;
            if (all & PF_BIT_DEAD) inf |= PF_INFO_DEAD;
            if (lower && border) inf |= PF_INFO_LPUB;
            if (!lower) inf &= ~(PF_INFO_LPUB | PF_INFO_LOW);
            a.info[T.tile] = inf;
            const uint32_t ended = asked + share - newly;
            if (ended) atomicAdd(&counts[PF_ENDED], ended);
        }
    }
}

// Wave 0 waits for work: takes down the flag of one of the workgroup's tiles
// and returns the tile with the flag's rows, or finds that the stage is over,
// or gives up (the abort words, or no progress of any workgroup for the wait
// bound; a bound of zero gives up at the first poll without work).
// Workgroup 0 finds out that the stage is over, for all: the others read one
// word a poll beside their flags.
__device__ inline int pf_poll(const PfArgs& a, uint32_t stage, uint32_t nown,
                              unsigned long long& rows) {
    const int lane = threadIdx.x & 63;
    uint32_t mine = lane < (int)nown ? pf_own(a, lane) : 0u;
    unsigned long long* fl = a.flags + (size_t)(stage & 1u) * a.total;
    uint32_t* over = &a.ctrl[CTL_PF_OVER];
    uint64_t t0 = wall_clock64();
    uint32_t seen = 0;
    for (uint32_t it = 1;; ++it) {
        const uint32_t o = ld(over);
        uint32_t found = ~0u;
        for (uint32_t j = 0; j < nown; j += 64) {
            if (nown > 64) mine = j + lane < nown ? pf_own(a, j + lane) : 0u;
            unsigned long long f = 0;
            if (j + lane < nown)
                f = __hip_atomic_load(fl + mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long m = __ballot(f != 0ull);
            if (m) {
                found = (uint32_t)__builtin_amdgcn_readlane((int)mine, __ffsll((long long)m) - 1);
                break;
            }
        }
        const uint32_t ov = (uint32_t)__builtin_amdgcn_readfirstlane((int)o);
        if (ov == PF_OVER_ABANDON) return PF_ABANDON;
        if (found != ~0u) {
            unsigned long long r = 0;
            if (lane == 0)
                r = __hip_atomic_exchange(fl + found, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)r);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(r >> 32));
            rows = ((unsigned long long)hi << 32) | lo;
            return (int)found;
        }
        if (ov > stage) return PF_DONE;
        if (blockIdx.x == 0) {
            const uint32_t ended = pf_sum(a, stage, PF_ENDED);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // the sums in this order
            if (ended == pf_sum(a, stage, PF_ASKED)) {
                if (lane == 0) st(over, stage + 1u);
                return PF_DONE;
            }
        }
        if (it % BAR_CHECK_EVERY == 0 || a.gb.limit == 0) {
            const uint32_t ended = pf_sum(a, stage, PF_ENDED);
            if (ended != seen && a.gb.limit != 0) {
                seen = ended;
                t0 = wall_clock64();
            }
            const bool give = bar_should_stop(a.gb, t0, it % BAR_HOST_EVERY == 0);
            if (__ballot(give)) {
                if (lane == 0) {
                    st(&a.gb.bar[BAR_ABORT], 1u);
                    st(over, PF_OVER_ABANDON);
                    atomicCAS(a.gb.status, 0u, (uint32_t)(-CAGEO_ERR_ABORTED));
                }
                return PF_ABANDON;
            }
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Solves the rows `rd` of the strip (and what they reach) in the tile held in
// LDS, in the lower bound also settles which undecided cells sit at their Z,
// and publishes the sides with cells lowered here or before (`lowered`).
__device__ inline void pf_solve(PfShared& S, PfTile& T, const PfArgs& a, const PfBlock& b,
                                uint32_t stage, uint32_t rd, uint32_t lowered, float floor,
                                float cfloor, uint32_t share, bool all_lower) {
    const uint32_t before = T.low;
    fill_sweeps(S, rd, T.zr, T.lower ? T.obst & ~T.dead : T.obst, lowered);
    T.chg |= lowered;
    if (T.lower) {
        const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        T.low = 0;
        for (int k = 0; k < STRIP; ++k) {  // undecided cells are few: most rows have none
            if (__ballot((T.dead >> k) & 1u) == 0) continue;
            if (((T.dead >> k) & 1u) &&
                !(S.rel[(strip * STRIP + k + 1) * HALO_W + lx + 1] > T.zr[k]))
                T.low |= 1u << k;
        }
        if (__ballot(T.low != before)) {
            const uint32_t now = wave_sum5((uint32_t)__popc(T.low));
            const uint32_t was = wave_sum5((uint32_t)__popc(before));
            if (lx == 0 && now != was)
                atomicAdd(&pf_own_counts(a, stage)[PF_LOW], now - was);
        }
    }
    pf_publish(S, T, a, b, stage, lowered, floor, cfloor, share, all_lower);
    __syncthreads();
}

// MULTI: a table of rasters (else the one raster of the arguments; two
// instantiations keep the one-raster code free of table lookups).
template <bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_pf_fill(PfArgs a) {
    __shared__ PfShared S;
    if (grid_aborted(a.gb)) return;
    float mn1 = 0.0f;
    bool ok1 = true;
    if (!MULTI) {
        ok1 = pf_raster_ok(a.one, mn1);
        if (!ok1) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *a.one.status = (uint32_t)(-CAGEO_ERR_RANGE);
            return;
        }
    }
    const int strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = gridDim.x;
    PfTile T;
    uint32_t nown = 0;              // the workgroup's blocks (a.own)
    uint32_t claimed = blockIdx.x;  // the block it takes next, in stage 0
    uint32_t undecided = ~0u;       // cells at their Z in the last lower bound
    bool last = false;  // this U stage only takes over the last L
    uint32_t stage = 0;
    for (;; ++stage) {
        const bool lower = stage & 1;
        // the words of the stage after the next (last used two stages ago,
        // which every workgroup has left: this one is past the stage between)
        if (blockIdx.x == 0 && threadIdx.x < CTL_PF_GROUPS) {
            uint32_t* c = pf_counts(a, stage + 2, threadIdx.x);
            st(&c[PF_ASKED], threadIdx.x == 0 ? G : 0u);
            st(&c[PF_ENDED], 0u);
            st(&c[PF_LOW], 0u);
        }
        // a lower bound left in LDS belongs to the stage that is over
        if (!lower && T.lower) {
            flush_tile<MULTI>(S, T, a, false, mn1, ok1);
            T.tile = -1;
            T.lower = false;
        }
        // Visits: first one to each of the workgroup's tiles that the stage
        // concerns, then those the neighbours ask for.  One body for both, and
        // so one copy of the sweeps: with three the loop outgrew the
        // instruction cache.  (The compiler keeps 293 of its scalars in vector
        // registers; in the table form 275, with 10 vector registers in
        // scratch.)
        uint32_t ahead = 0;
        bool began = false;
        for (;;) {
            const bool first = stage == 0 ? claimed < a.total : ahead < nown;
            uint32_t t, inf = 0;
            unsigned long long rows = 0;
            if (first) {
                if (stage == 0) {
                    t = claimed;
                    if (threadIdx.x == 0) a.own[(size_t)nown * G + blockIdx.x] = (int)t;
                    ++nown;
                } else {
                    t = pf_own(a, ahead++);
                }
                if (stage > 0) {
                    inf = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.info[t]);
                    if (!(inf & (lower ? PF_INFO_DEAD : PF_INFO_DEAD | PF_INFO_LPUB))) {
                        if (!lower && threadIdx.x == 0) a.info[t] = inf & ~PF_INFO_LOW;
                        continue;
                    }
                }
            } else {
                if (!began) {  // the first visits are over
                    wait_stores();
                    __syncthreads();
                    if (threadIdx.x == 0) atomicAdd(&pf_own_counts(a, stage)[PF_ENDED], 1u);
                    began = true;
                }
                if (threadIdx.x < 64) {
                    const int cmd = pf_poll(a, stage, nown, rows);
                    if (threadIdx.x == 0) {
                        S.cmd = cmd;
                        S.rows_lo = (uint32_t)rows;
                        S.rows_hi = (uint32_t)(rows >> 32);
                    }
                }
                __syncthreads();
                const int cmd = __builtin_amdgcn_readfirstlane(S.cmd);
                rows = ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)S.rows_hi) << 32) |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)S.rows_lo);
                __syncthreads();
                if (cmd == PF_ABANDON) return;
                if (cmd == PF_DONE) break;
                t = (uint32_t)cmd;
                if (lower) inf = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.info[t]);
            }
            const PfBlock b = pf_block<MULTI>(a, t, mn1, ok1);
            uint32_t next = a.total;
            if (MULTI && !b.ok) {
                // a raster outside the domain: its blocks have no work, now or
                // later (they come here once, when claimed)
                if (threadIdx.x == 0) {
                    a.info[t] = 0u;
                    if (b.lb == 0) *b.R.status = (uint32_t)(-CAGEO_ERR_RANGE);
                    if (nown < a.most) next = G + atomicAdd(&a.ctrl[CTL_PF_CLAIM], 1u);
                    S.cmd = (int)next;
                }
                __syncthreads();
                claimed = (uint32_t)__builtin_amdgcn_readfirstlane(S.cmd);
                __syncthreads();
                continue;
            }
            // ---- the tile into LDS: the upper bound, or the lower bound where
            // LDS holds it since this stage
            const bool fresh = first && stage == 0;
            if (T.tile != (int)t || (T.lower && !lower)) {
                flush_tile<MULTI>(S, T, a, lower, mn1, ok1);
                if (!fresh) load_again(S, T, a, b, t, lower && !first && (inf & PF_INFO_LOW));
            } else if (lower && !T.lower) {
                flush_tile<MULTI>(S, T, a, lower, mn1, ok1);  // LDS goes on as the lower bound
            }
            visit_reset(S);
            uint32_t share = first ? 0u : 1u, seeds = 0;
            if (fresh) {
                T.tile = (int)t;
                // a flag raised so far is answered by this visit: taken down
                // before the ring is read
                if (threadIdx.x == 0) {
                    a.info[t] = 0u;
                    S.cmd = __hip_atomic_exchange(a.flags + t, 0ull, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT) != 0ull;
                }
                __syncthreads();
                share = (uint32_t)__builtin_amdgcn_readfirstlane(S.cmd);
                seeds = load_first(S, T, b);
                put_floors(T, a);
            }
            float floor, cfloor;  // of this thread's ring cell and corner
            const bool any = load_ring(S, a, b, stage, lower && !first, floor, cfloor) || seeds != 0u;
            if (lower && !first && !T.lower) {
                // a tile without undecided cells, changed by its neighbours
                T.lower = true;
            }
            const bool go = __syncthreads_or(any);
            uint32_t due = strip_rows(rows, strip);
            if (fresh) {
                due = go ? 0xffffffffu : 0u;  // nothing has reached it yet: nothing to solve
            } else if (first && lower) {
                // undecided cells whose relays now prove them blocked are settled
                const int lx = threadIdx.x & 63;
                uint32_t keep = 0, dr = 0;
                for (int k = 0; k < STRIP; ++k) {
                    if (__ballot((T.dead >> k) & 1u) == 0) continue;
                    bool c = false;
                    if ((T.dead >> k) & 1u)
                        c = min8(S.rel, (strip * STRIP + k + 1) * HALO_W + lx + 1) > T.zr[k];
                    if (c) keep |= 1u << k;
                    if (__ballot(c)) dr |= 1u << k;
                }
                due = dr | (dr << 16);
                T.dead = keep;
                T.low = 0;
                T.lower = true;
                T.chg |= keep;    // their written-back value is Z
                __syncthreads();  // the relays above are read before one is lowered
            } else if (first) {
                // those above their Z in the lower bound relay for good
                const uint32_t sure = T.dead & ~T.low;
                uint32_t dr = 0;
                for (int k = 0; k < STRIP; ++k)
                    if (__ballot((sure >> k) & 1u)) dr |= 1u << k;
                due = dr | (dr << 16);
                T.obst &= ~sure;
                T.dead = T.low;
                T.low = 0;
                T.chg |= sure;
            }
            // the next claim is under way during the visit
            if (fresh && threadIdx.x == 0 && nown < a.most) next = G + atomicAdd(&a.ctrl[CTL_PF_CLAIM], 1u);
            pf_solve(S, T, a, b, stage, due, seeds, floor, cfloor, share,
                     first && !lower && (inf & PF_INFO_LPUB) != 0u);
            if (fresh) {
                if (threadIdx.x == 0) S.cmd = (int)next;
                __syncthreads();
                claimed = (uint32_t)__builtin_amdgcn_readfirstlane(S.cmd);
                __syncthreads();
            }
        }
        if (last) break;
        if (lower) {
            const uint32_t low = pf_sum(a, stage, PF_LOW);
            if (low == 0u) {
                // the lower bound is the result; with one tile a workgroup it
                // is in LDS wherever it differs from the upper bound
                if (a.most == 1) break;
                last = true;
            } else if (low >= undecided) {
                // (every pair of stages settles a cell: not to be reached)
                if (blockIdx.x == 0 && threadIdx.x == 0)
                    a.ctrl[CTL_STATUS] = (uint32_t)(-CAGEO_ERR_NOT_CONVERGED);
                return;
            }
            undecided = low;
        }
    }
    // ---- the result: the tile in LDS, and in the tiles written back before,
    // Z where nothing came
    for (uint32_t j = 0; j < nown; ++j) {
        const uint32_t t = pf_own(a, j);
        const PfBlock b = pf_block<MULTI>(a, t, mn1, ok1);
        if (MULTI && !b.ok) continue;
        if (T.tile == (int)t) {
            write_cells(S, T, b, true);
        } else if (__builtin_amdgcn_readfirstlane((int)a.info[t]) & PF_INFO_INF) {
            const PfRaster& R = b.R;
            const int x = (b.lb % R.ntx) * TILE + (threadIdx.x & 63);
            const int y0 = (b.lb / R.ntx) * TILE + strip * STRIP;
            for (int k = 0; k < STRIP; ++k) {
                if (x >= R.W || y0 + k >= R.H) continue;
                const size_t gi = (size_t)(y0 + k) * R.W + x;
                if (!(R.w[gi] < PF_INF)) R.w[gi] = R.zq[gi];
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.ctrl[CTL_ROUNDS] = (stage + 1) / 2;  // lower bounds taken
        a.ctrl[CTL_PASSES] = stage + 1;        // stages
    }
}

// State of a launch of `G` workgroups: no flag up, no side relays, no floor
// known, the stage counters.
__global__ __launch_bounds__(256) void k_pf_start(PfArgs a, uint32_t G) {
    const size_t n = (size_t)a.total;
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = i0; i < 2 * n; i += stride) a.flags[i] = 0ull;
    for (size_t i = i0; i < PF_PLANES * n * PF_SIDES / 4; i += stride) {
        const float v = i < PF_FLOOR * n * PF_SIDES / 4 ? PF_INF : 0.0f;
        reinterpret_cast<float4*>(a.xb)[i] = make_float4(v, v, v, v);
    }
    for (size_t i = i0; i < 4 * CTL_PF_STAGE; i += stride)
        a.ctrl[CTL_PF_COUNTS + i] = i % CTL_PF_STAGE == PF_ASKED ? G : 0u;
    if (i0 == 0) {
        a.ctrl[CTL_PF_OVER] = 0u;
        a.ctrl[CTL_PF_CLAIM] = 0u;
    }
}

PfRaster pf_raster(Context* c, const float* zq, float* w, float nodata) {
    PfRaster R;
    R.zq = zq;
    R.w = w;
    R.low = reinterpret_cast<float*>(c->d_dist);  // the routing's distances: idle here
    R.W = c->W;
    R.H = c->H;
    R.ntx = c->ntx;
    R.nty = c->nty;
    R.nodata = nodata;
    R.scal = c->d_scal;
    R.status = c->d_ctrl + CTL_STATUS;
    return R;
}

int occupancy_cap(const void* fn, int device, int* cap) {
    int per_cu = 0;
    CAGEO_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, TILE_THREADS, 0));
    hipDeviceProp_t prop;
    CAGEO_HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (per_cu < 1) return CAGEO_ERR_HIP;
    *cap = per_cu * prop.multiProcessorCount;
    return CAGEO_OK;
}

// Both launches of a fill.  Ordinary launches: the workgroups wait for each
// other's work, so all must run at once, which the occupancy cap on the grid
// guarantees (work of other kernels on the device can only delay the start of
// some).  Cooperative launches are not used: the runtime allows them to one
// process at a time.  No more workgroups than blocks: with one block each, a
// tile stays in its workgroup's LDS from the first visit to the result.
template <bool MULTI>
int pf_launch(PfArgs& a, int cap, hipStream_t s) {
    const uint32_t G = std::min<uint32_t>((uint32_t)cap, a.total);
    // twice an even share: a workgroup with easy blocks takes more of them
    a.most = a.total <= G ? 1u : 2u * ((a.total + G - 1) / G);
    const int init = (int)std::min<uint32_t>(1024u, (a.total + 1u) / 2u);
    hipLaunchKernelGGL(k_pf_start, dim3(init), dim3(256), 0, s, a, G);
    CAGEO_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_pf_fill<MULTI>, dim3(G), dim3(TILE_THREADS), 0, s, a);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

}  // namespace

// Co-resident workgroups of the persistent kernel on this device.
int pit_fill_grid_cap(Context* c, int* cap) {
    return occupancy_cap(reinterpret_cast<const void*>(k_pf_fill<false>), c->device, cap);
}

int pit_fill_persistent_grid(Context* c, int* grid) {
    if (c->pf_grid <= 0) CAGEO_TRY(pit_fill_grid_cap(c, &c->pf_grid));
    *grid = c->pf_grid;
    return CAGEO_OK;
}

int pit_fill_quantized(Context* c, float* zq, float* w, float nodata) {
    int grid = 0;
    CAGEO_TRY(pit_fill_persistent_grid(c, &grid));
    PfArgs a;
    a.one = pf_raster(c, zq, w, nodata);
    a.rs = nullptr;
    a.bmap = nullptr;
    a.total = (uint32_t)c->ntiles;
    a.flags = reinterpret_cast<unsigned long long*>(c->d_rows);
    a.own = c->d_work3;  // (7 words a block, idle here)
    a.xb = c->d_xb;
    a.masks = c->d_pfmask;
    a.info = c->d_pfinfo;
    a.ctrl = c->d_ctrl;
    a.gb = context_gridbar(c);
    return pf_launch<false>(a, grid, c->stream);
}

// Raster table of a batch: each context's d_z -> d_w with its DEM nodata.
int pit_fill_tables(MultiState* m, Context* const* ctxs) {
    std::vector<PfRaster> t(m->nr);
    for (int r = 0; r < m->nr; ++r) t[r] = pf_raster(ctxs[r], ctxs[r]->d_z, ctxs[r]->d_w, ctxs[r]->nodata_dem);
    CAGEO_HIP_TRY(hipMalloc(&m->d_pf, t.size() * sizeof(PfRaster)));
    CAGEO_HIP_TRY(hipMemcpy(m->d_pf, t.data(), t.size() * sizeof(PfRaster), hipMemcpyHostToDevice));
    CAGEO_TRY(occupancy_cap(reinterpret_cast<const void*>(k_pf_fill<true>),
                            ctxs[0]->device, &m->pf_cap));
    if (m->pf_grid <= 0) m->pf_grid = m->pf_cap;
    return CAGEO_OK;
}

int pit_fill_multi(MultiState* m, hipStream_t s) {
    PfArgs a;
    a.one = PfRaster{};
    a.rs = static_cast<const PfRaster*>(m->d_pf);
    a.bmap = m->d_bmap;
    a.total = (uint32_t)m->total;
    a.flags = reinterpret_cast<unsigned long long*>(m->d_rows);
    a.own = m->d_work;  // (7 words a block, idle here)
    a.xb = m->d_xb;
    a.masks = m->d_pfmask;
    a.info = m->d_pfinfo;
    a.ctrl = m->d_ctrl;
    a.gb = multi_gridbar(m);
    return pf_launch<true>(a, m->pf_grid, s);
}

}  // namespace cageo
