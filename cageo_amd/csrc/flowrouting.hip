// Flow routing: FlowRoutingAlgorithm<T,U>::execute, FlowRoutingAlgorithm.h:
// 69-94; parity target FlowRoutingAlgorithm_CPU_OpenMP (D8 :53-151, flats
// :153-249 of FlowRoutingAlgorithmCPUOpenMP.h).
//
// D8: edge cells point out of the grid; cells at 0 are stream cells with no
// direction; otherwise the steepest of N, NE, E, SE, S, SW, W, NW with
// drop = z_c - z_n, diagonal drops divided by 1.41421356237309505f, strict
// '>' so the first of equal drops wins.  A cell with no positive drop is
// flat.
//
// Flats: the reference resolves them in rounds k = -1, 1, 2, ...: a flat c
// takes every neighbour n (same order, the last one wins) with
// flatDist[n] == k and z_n <= z_c.  That is a breadth-first distance
//   d(c) = 1 + min { d(n) : n an 8-neighbour, z_n <= z_c,
//                            n has a direction (d = 0) or is a flat },
// followed by direction = last n in order with d(n) = d(c) - 1 and
// z_n <= z_c.  d is computed tile by tile: inside a 64x64 tile by the search
// itself, a whole level of it in a few instructions (flat_levels), and
// between tiles by passes over the tiles whose ring changed.
#include <algorithm>
#include <vector>

#include "tiles.hpp"

namespace cageo {

namespace {

constexpr int D_INF = 0x3fffffff;
constexpr int D_STREAM = -2;
constexpr int D_OUT = -3;

__device__ constexpr int FDX[8] = {0, 1, 1, 1, 0, -1, -1, -1};
__device__ constexpr int FDY[8] = {-1, -1, 0, 1, 1, 1, 0, -1};

typedef unsigned long long Row64;  // a bit per cell of a tile's row, bit = column

constexpr int FR_D = HALO_W * HALO_W;  // distances of a tile and its ring
constexpr int FR_PLANES = 8;
constexpr int FR_STEPS = (1 << FR_PLANES) - 1;  // levels a run of flat_levels records

// A tile's distances and the record of a run of flat_levels: the step that
// set a cell is the number whose bits the planes hold there (0: none).
struct FrSolve {
    Row64 plane[FR_PLANES][TILE];
    int lvl[FR_STEPS + 1];  // distance that a step gave
};
struct FrTile {
    int d[FR_D];
    Row64 inf[TILE], aux[TILE];  // flats without a distance; see flat_solve
    int steps, more;             // of the last run: steps taken; levels are left
    uint32_t bits;               // neighbour tiles concerned
    uint32_t pushed;             // tiles this workgroup listed in the pass (thread 0's)
};

// One raster of a launch.
struct FrRaster {
    const float* z;
    int8_t* fd;
    int32_t* dist;
    Row64* nbr;  // per block: 4 directions x 64 rows (see fr_nbr)
    int W, H, ntx, nty;
};

// A launch over one raster (`one`, rs null) or over the rasters of a
// table, whose 64x64 blocks are numbered globally (bmap).
struct FrArgs {
    FrRaster one;
    const FrRaster* __restrict__ rs;
    const int2* __restrict__ bmap;  // per block: (raster, block within it)
    int total;
    int* work;      // 3 lists of `total` entries
    uint32_t* mark; // per-block epoch stamps
    Row64* nbr;     // per block: the other 4 directions x 64 rows
    uint32_t* ctrl;
    GridBar gb;     // grid barrier
    int max_passes;
};

struct FrBlock {
    FrRaster R;
    int lb, gbase;
};
template <bool MULTI>
__device__ inline FrBlock fr_block(const FrArgs& a, int g) {
    FrBlock b;
    g = __builtin_amdgcn_readfirstlane(g);
    if constexpr (!MULTI) {
        b.R = a.one;
        b.gbase = 0;
    } else {
        const int2 m = a.bmap[g];
        const int r = __builtin_amdgcn_readfirstlane(m.x);
        b.gbase = g - __builtin_amdgcn_readfirstlane(m.y);
        b.R = a.rs[r];
    }
    b.lb = g - b.gbase;
    return b;
}

// The neighbour masks of a block for direction q: row r's word has bit x set
// where cell (x, r) is a flat and its neighbour in direction q (in the tile
// or its ring) is not higher.  A byte a cell in two buffers of four
// directions each that the stages around this one use (the border tables of
// the tracing, the wall masks of the pit fill).
__device__ inline Row64* fr_nbr(const FrArgs& a, const FrBlock& b, int q) {
    return (q < 4 ? b.R.nbr + (size_t)b.lb * (4 * TILE)
                  : a.nbr + (size_t)(b.gbase + b.lb) * (4 * TILE)) + (q & 3) * TILE;
}

__device__ inline uint32_t ld(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// s / 1.41421356237309505f for s in [2^-77, 2^100), correctly rounded:
// Markstein's correction of a quotient by its exact remainder (equal to the
// division for every significand), three instructions where the division
// takes eleven.
constexpr float DIAGONAL = 1.41421356237309505f;
constexpr float DIV_LOW = 0x1p-77f, DIV_HIGH = 0x1p100f;
__device__ inline float over_diagonal(float s) {
    constexpr float y = 1.0f / DIAGONAL;
    const float q = s * y;
    return __builtin_fmaf(__builtin_fmaf(-q, DIAGONAL, s), y, q);
}

// D8 of one cell (FlowRoutingAlgorithmCPUOpenMP.h:60-150) at grid position
// (x, y), its elevation zc and its neighbours' nb.  Returns the initial
// distance: 0 has a direction, D_STREAM, or D_INF (flat); `dir` the
// direction, x offset in the low byte and y offset in the next.  Edge cells
// point out of the grid and read no neighbour, so values outside the grid
// are never used.  Without branches but for drops outside the range of
// over_diagonal (a test and a division behind it for each neighbour took the
// launch 38 us at 1000 x 777 and 157 at 4096^2; now 34 and 143).
__device__ inline int32_t d8_of(float zc, const float* nb, int x, int y, int W, int H,
                                uint32_t& dir) {
    float s[8], steepest = 0.0f, most = 0.0f;
    uint32_t least = 0xffffffffu;  // of the positive diagonal drops, less one
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        s[k] = fmaxf(zc - nb[k], 0.0f);  // (0 for a NaN)
        if (k & 1) {
            most = fmaxf(most, s[k]);
            least = min(least, __float_as_uint(s[k]) - 1u);
        }
    }
    if (most >= DIV_HIGH || least < __float_as_uint(DIV_LOW) - 1u) {
#pragma unroll
        for (int k = 1; k < 8; k += 2) s[k] = s[k] / DIAGONAL;
    } else {
#pragma unroll
        for (int k = 1; k < 8; k += 2) s[k] = over_diagonal(s[k]);
    }
    dir = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t code = (uint32_t)(uint8_t)FDX[k] | (uint32_t)(uint8_t)FDY[k] << 8;
        dir = s[k] > steepest ? code : dir;
        steepest = fmaxf(steepest, s[k]);
    }
    int32_t d = steepest > 0.0f ? 0 : D_INF;
    d = zc == 0.0f ? D_STREAM : d;
    dir = zc == 0.0f ? 0u : dir;
    const int dxi = x == 0 ? -1 : x == W - 1 ? 1 : 0, dyi = y == 0 ? -1 : y == H - 1 ? 1 : 0;
    if ((dxi | dyi) != 0) {
        d = 0;
        dir = (uint32_t)(uint8_t)dxi | (uint32_t)(uint8_t)dyi << 8;
    }
    return d;
}

__device__ inline Row64 row_prev(Row64 v) {  // the row above's word (none above the first)
    const uint32_t lo = (uint32_t)dpp_i<DPP_WAVE_SHR1>(0, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)dpp_i<DPP_WAVE_SHR1>(0, (int)(uint32_t)(v >> 32));
    return ((Row64)hi << 32) | lo;
}
__device__ inline Row64 row_next(Row64 v) {
    const uint32_t lo = (uint32_t)dpp_i<DPP_WAVE_SHL1>(0, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)dpp_i<DPP_WAVE_SHL1>(0, (int)(uint32_t)(v >> 32));
    return ((Row64)hi << 32) | lo;
}
__device__ inline Row64 row_read(Row64 v, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return ((Row64)hi << 32) | lo;
}
__device__ inline void row_write(Row64& v, Row64 x, int lane) {
    v = (int)(threadIdx.x & 63) == lane ? x : v;
}
__device__ inline int wave_min(int v) {
    int none = 0;
    auto least = [](int& s, int&, int p, int) { s = min(s, p); };
    CAGEO_SCAN_UP(dpp_i, v, none, (int)D_INF, 0, least);
    return lane_read(v, 63);
}

// The breadth-first search of a tile as one wave holds it: lane r has row r
// of the frontier, the masks and the distances that come in from the ring.
struct Levels {
    Row64 nbr[8];  // neighbour masks (fr_nbr)
    Row64 front;   // cells of distance `level` whose neighbours come next
    Row64 inf;     // flats without a distance
    Row64 fin;     // flats with one that has not been compared yet
    int level;
    int west, east;    // distance the ring offers the row's first and last cell
    int north, south;  // ... and cell `lane` of the first and last row
    int next;          // least of those
};

// Best distance of cell c (offset in the tile's distances) by its ring
// neighbours in directions q0..q2 (`m` bit 0..2: not higher), D_INF where it
// is none or no better than the cell's own.
__device__ inline int ring_offer(const int* d, int c, int q0, int q1, int q2, uint32_t m) {
    const int n0 = d[c + FDY[q0] * HALO_W + FDX[q0]], n1 = d[c + FDY[q1] * HALO_W + FDX[q1]],
              n2 = d[c + FDY[q2] * HALO_W + FDX[q2]];
    int v = D_INF;
    if ((m & 1u) && n0 >= 0) v = min(v, n0 + 1);
    if ((m & 2u) && n1 >= 0) v = min(v, n1 + 1);
    if ((m & 4u) && n2 >= 0) v = min(v, n2 + 1);
    return v < d[c] ? v : D_INF;
}
__device__ inline uint32_t bit3(Row64 a, Row64 b, Row64 c, int x) {
    return ((uint32_t)(a >> x) & 1u) | (((uint32_t)(b >> x) & 1u) << 1) |
           (((uint32_t)(c >> x) & 1u) << 2);
}
__device__ inline void ring_offers(Levels& v, const int* d) {
    const int lane = threadIdx.x & 63;
    const Row64* n = v.nbr;
    v.west = ring_offer(d, (lane + 1) * HALO_W + 1, 5, 6, 7, bit3(n[5], n[6], n[7], 0));
    v.east = ring_offer(d, (lane + 1) * HALO_W + TILE, 1, 2, 3, bit3(n[1], n[2], n[3], TILE - 1));
    const Row64 n7 = row_read(n[7], 0), n0 = row_read(n[0], 0), n1 = row_read(n[1], 0);
    v.north = ring_offer(d, HALO_W + lane + 1, 7, 0, 1, bit3(n7, n0, n1, lane));
    const Row64 s3 = row_read(n[3], TILE - 1), s4 = row_read(n[4], TILE - 1),
                s5 = row_read(n[5], TILE - 1);
    v.south = ring_offer(d, TILE * HALO_W + lane + 1, 3, 4, 5, bit3(s3, s4, s5, lane));
    v.next = wave_min(min(min(v.west, v.east), min(v.north, v.south)));
}

// A run of the search by the first wave: levels in order until none is left
// or FR_STEPS of them have set cells.  A level takes the cells beside the
// frontier, all 4096 at once, and those to which the ring offers it.  A cell
// that had a distance is compared with the first level that reaches it: a
// later one is no better.
// (A front along a row meets 64 of them in one lane: such rows are compared by
// the whole wave.  With all of them cell by cell, a wide flat whose tiles the
// distances cross more than once, a constant 1100 x 1100, took 1549 us to
// route, 489 now.)
// A chain of levels, each about 100 vector instructions of one wave, bounds
// it; the step numbers are recorded in bit planes because a store a cell
// would cost the fullest row's cells one after the other.  Sweeps of row
// solves (min-plus scans along each row, four waves a tile) did the same
// work before: the D8 kernel took 81 us at 1000 x 777 and 313 at 4096^2, then
// 38 and 157; the passes 117 and 379, now 87 and 307 (a grid barrier a
// pass, some 8 to 13 us, is most of what is left of them).
__device__ inline void flat_levels(Levels& v, FrTile& T, FrSolve& S) {
    const int lane = threadIdx.x & 63;
    Row64 plane[FR_PLANES];
#pragma unroll
    for (int j = 0; j < FR_PLANES; ++j) plane[j] = 0;
    int steps = 0;
    bool more = true;
    while (steps < FR_STEPS) {
        Row64 c = 0;
        if (__ballot(v.front != 0)) {
            ++v.level;
            const Row64 up = row_prev(v.front), dn = row_next(v.front), f = v.front;
            c = (up & v.nbr[0]) | ((up >> 1) & v.nbr[1]) | ((f >> 1) & v.nbr[2]) |
                ((dn >> 1) & v.nbr[3]) | (dn & v.nbr[4]) | ((dn << 1) & v.nbr[5]) |
                ((f << 1) & v.nbr[6]) | ((up << 1) & v.nbr[7]);
        } else {
            if (v.next == D_INF) {
                more = false;
                break;
            }
            v.level = v.next;
        }
        if (v.level == v.next) {
            const int l = v.level;
            const Row64 north = __ballot(v.north == l), south = __ballot(v.south == l);
            if (v.west == l) c |= 1ull;
            if (v.east == l) c |= 1ull << (TILE - 1);
            if (lane == 0) c |= north;
            if (lane == TILE - 1) c |= south;
            if (v.west == l) v.west = D_INF;
            if (v.east == l) v.east = D_INF;
            if (v.north == l) v.north = D_INF;
            if (v.south == l) v.south = D_INF;
            v.next = wave_min(min(min(v.west, v.east), min(v.north, v.south)));
        }
        Row64 set = c & v.inf;
        Row64 old = c & v.fin;
        v.inf &= ~set;
        v.fin &= ~old;
        if (__ballot(old != 0)) {
            constexpr int OLD_FEW = 4;  // of a row: compared cell by cell
            for (Row64 many = __ballot(__popcll(old) > OLD_FEW); many != 0; many &= many - 1) {
                const int r = __builtin_ctzll(many);
                const Row64 better =
                    __ballot(T.d[(r + 1) * HALO_W + lane + 1] > v.level) & row_read(old, r);
                row_write(set, set | better, r);
                row_write(old, 0ull, r);
            }
            while (__ballot(old != 0)) {
                if (old != 0) {
                    const int x = __builtin_ctzll(old);
                    old &= old - 1;
                    if (T.d[(lane + 1) * HALO_W + x + 1] > v.level) set |= 1ull << x;
                }
            }
        }
        v.front = set;
        if (__ballot(set != 0)) {
            ++steps;
#pragma unroll
            for (int j = 0; j < FR_PLANES; ++j)
                plane[j] |= set & (0ull - (Row64)((steps >> j) & 1));
            S.lvl[steps] = v.level;
        }
    }
#pragma unroll
    for (int j = 0; j < FR_PLANES; ++j) S.plane[j][lane] = plane[j];
    if (lane == 0) {
        T.steps = steps;
        T.more = more;
    }
}

// The flat distances of a tile, given its ring's: T.d lowered to them.
// T.inf holds the flats without a distance and T.aux, in a tile's first
// solve, the cells of distance 0, later the flats that have one (the tile
// is then at the fixed point of its last solve, so what changes starts at
// the ring).  Returns the changed cells of the thread's column, bit = row of
// its strip.  Called after a barrier that follows the writes of T.
__device__ inline uint32_t flat_solve(Levels& v, FrTile& T, FrSolve& S, bool first) {
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (strip == 0) {
        v.inf = T.inf[lx];
        const Row64 aux = T.aux[lx];
        v.front = first ? aux : 0ull;
        v.fin = first ? 0ull : aux;
        v.level = 0;
        ring_offers(v, T.d);
    }
    uint32_t changed = 0;
    for (;;) {
        if (strip == 0) flat_levels(v, T, S);
        __syncthreads();
        const int steps = __builtin_amdgcn_readfirstlane(T.steps);
        const bool more = __builtin_amdgcn_readfirstlane(T.more) != 0;
        const int planes = 32 - __builtin_clz(steps | 1);
        if (steps) {
            uint32_t s[STRIP];
#pragma unroll
            for (int k = 0; k < STRIP; ++k) s[k] = 0;
            for (int j = 0; j < planes; ++j) {
#pragma unroll
                for (int k = 0; k < STRIP; ++k)
                    s[k] |= ((uint32_t)(S.plane[j][strip * STRIP + k] >> lx) & 1u) << j;
            }
#pragma unroll
            for (int k = 0; k < STRIP; ++k)
                if (s[k]) {
                    T.d[(strip * STRIP + k + 1) * HALO_W + lx + 1] = S.lvl[s[k]];
                    changed |= 1u << k;
                }
        }
        if (!more) break;
        __syncthreads();
    }
    return changed;
}

// After a solve: the changed distances of the tile written back (with
// write_all all of them), and the neighbour tiles that a changed border cell
// concerns listed for the next pass: those with a flat beside it, in this
// tile's ring, whose distance as loaded exceeds the cell's plus one (two
// flats side by side are equally high, so the flat can take it; distances
// only decrease, so this errs towards listing).
__device__ inline void flat_finish(FrTile& T, const FrArgs& args, const FrBlock& b, int tx, int ty,
                                   uint32_t changed, bool write_all, int* work_out,
                                   uint32_t* count_out, uint32_t epoch) {
    const FrRaster& R = b.R;
    const int x0 = tx * TILE, y0 = ty * TILE;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const int ly = strip * STRIP + k;
        const bool in = x0 + lx < R.W && y0 + ly < R.H;
        if (in && (write_all || (changed & (1u << k))))
            R.dist[(size_t)(y0 + ly) * R.W + x0 + lx] = T.d[(ly + 1) * HALO_W + lx + 1];
    }
    uint32_t bits = 0;
    const uint32_t edge = (lx == 0 || lx == TILE - 1)
                              ? 0xffffu
                              : ((strip == 0 ? 1u : 0u) |
                                 (strip == TILE_THREADS / 64 - 1 ? 1u << (STRIP - 1) : 0u));
    uint32_t cand = changed & edge;
    while (cand) {
        const int k = __builtin_ctz(cand);
        cand &= cand - 1;
        const int ly = strip * STRIP + k;
        const int li = (ly + 1) * HALO_W + lx + 1;
        const int cv = T.d[li];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int nx = lx + FDX[q], ny = ly + FDY[q];
            if (nx >= 0 && ny >= 0 && nx < TILE && ny < TILE) continue;
            const int nv = T.d[li + FDY[q] * HALO_W + FDX[q]];
            if (nv >= 1 && nv > cv + 1)
                bits |= 1u << tile_dir(nx < 0 ? -1 : (nx >= TILE ? 1 : 0),
                                       ny < 0 ? -1 : (ny >= TILE ? 1 : 0));
        }
    }
    bits = wave_or8(bits);
    if (lx == 0 && bits) atomicOr(&T.bits, bits);
    __syncthreads();
    if (strip == 0 && T.bits)  // uniform within the first wave
        activate_tiles(T.bits, tx, ty, R.ntx, R.nty, b.gbase, work_out, count_out, args.mark, epoch,
                       nullptr, 0, 0, 0, nullptr, nullptr, &T.pushed);
    __syncthreads();
}

// A listed tile of a flat pass: its distances with the ring and its
// neighbour masks loaded, then solved.
__device__ void bfs_tile(FrTile& T, FrSolve& S, const FrArgs& args, const FrBlock& b, int* work_out,
                         uint32_t* count_out, uint32_t epoch) {
    const FrRaster& R = b.R;
    const int tx = b.lb % R.ntx, ty = b.lb / R.ntx;
    const int x0 = tx * TILE, y0 = ty * TILE;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Levels v;
    {
        constexpr int ITER = (FR_D + TILE_THREADS - 1) / TILE_THREADS;
        int d[ITER];
#pragma unroll
        for (int j = 0; j < ITER; ++j) {  // all loads first (a cell outside loads cell 0)
            const int k = threadIdx.x + j * TILE_THREADS;
            const int hy = k / HALO_W, hx = k - hy * HALO_W;
            const int gx = x0 - 1 + hx, gy = y0 - 1 + hy;
            const bool in = k < FR_D && gx >= 0 && gy >= 0 && gx < R.W && gy < R.H;
            d[j] = R.dist[in ? (size_t)gy * R.W + gx : 0];
            if (!in) d[j] = D_OUT;
        }
        if (strip == 0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) v.nbr[q] = fr_nbr(args, b, q)[lx];
        }
#pragma unroll
        for (int j = 0; j < ITER; ++j) {
            const int k = threadIdx.x + j * TILE_THREADS;
            if (k < FR_D) T.d[k] = d[j];
        }
    }
    if (threadIdx.x == 0) T.bits = 0;
    __syncthreads();
    Row64 inf = 0, fin = 0;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const int d = T.d[(strip * STRIP + k + 1) * HALO_W + lx + 1];
        row_write(inf, __ballot(d == D_INF), k);
        row_write(fin, __ballot(d >= 1 && d < D_INF), k);
    }
    if (lx < STRIP) {
        T.inf[strip * STRIP + lx] = inf;
        T.aux[strip * STRIP + lx] = fin;
    }
    __syncthreads();
    const uint32_t changed = flat_solve(v, T, S, false);
    flat_finish(T, args, b, tx, ty, changed, false, work_out, count_out, epoch);
}

// The epoch stamp of pass 0's listings (the D8 kernel's); pass p lists with
// FR_EPOCH0 + p.  k_fr_reset clears every stamp to 0 before a launch, so the
// epochs can start over each launch and never come round to 0.
constexpr uint32_t FR_EPOCH0 = 1u;

// Before a launch's D8 kernel: every block's epoch stamp cleared (an
// abandoned launch may have left some, and the D8 kernel's blocks list each
// other, so none can clear its own there) and the worklist counts zeroed.
__global__ void k_fr_reset(FrArgs a) {
    for (int g = blockIdx.x * blockDim.x + threadIdx.x; g < a.total; g += gridDim.x * blockDim.x) {
        a.mark[g] = 0u;
    }
    if (blockIdx.x == 0) {
        if (threadIdx.x < 3) a.ctrl[CTL_COUNT + threadIdx.x] = 0u;
        if (threadIdx.x == 3) a.ctrl[CTL_FR_DONE] = 0u;
    }
}

// D8 and the first flat pass, one workgroup per block.  The block's
// elevations with a two-cell halo are staged in LDS, D8 is worked out for
// the 66 x 66 cells of its distance tile (its own and the ring around it:
// the ring's are the initial distances its neighbours start from) and with
// it the neighbour masks; the first pass solves the tile against that ring;
// then the block's distances go out, and the tiles its changed border cells
// concern are listed for pass 1 (list 1, epoch FR_EPOCH0).  The persistent
// kernel goes on from pass 1.
template <bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_fr_d8(FrArgs a) {
    constexpr int ZW = HALO_W + 2, ZN = ZW * ZW;  // elevations with two halo cells
    __shared__ FrTile T;
    __shared__ union {
        float zt[ZN];
        struct {
            Row64 nbr[8][TILE];
            FrSolve S;
        } s;  // once D8 is done
    } U;
    const FrBlock b = fr_block<MULTI>(a, blockIdx.x);
    const FrRaster& R = b.R;
    const int tx = b.lb % R.ntx, ty = b.lb / R.ntx;
    const int x0 = tx * TILE, y0 = ty * TILE;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    {
        constexpr int IT = (ZN + TILE_THREADS - 1) / TILE_THREADS;
        float v[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {  // all loads first (a cell outside loads cell 0)
            const int k = threadIdx.x + j * TILE_THREADS;
            const int hy = k / ZW, hx = k - hy * ZW;
            const int gx = x0 - 2 + hx, gy = y0 - 2 + hy;
            const bool in = k < ZN && gx >= 0 && gy >= 0 && gx < R.W && gy < R.H;
            v[j] = R.z[in ? (size_t)gy * R.W + gx : 0];
            if (!in) v[j] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const int k = threadIdx.x + j * TILE_THREADS;
            if (k < ZN) U.zt[k] = v[j];
        }
    }
    if (threadIdx.x == 0) {
        T.bits = 0;
        T.pushed = 0;
    }
    __syncthreads();
    // The ring, a cell a thread.
    for (int i = threadIdx.x; i < 4 * (HALO_W - 1); i += TILE_THREADS) {
        const int side = i / (HALO_W - 1), p = i - side * (HALO_W - 1);
        const int hx = side == 0 ? p : side == 1 ? HALO_W - 1 : side == 2 ? HALO_W - 1 - p : 0;
        const int hy = side == 0 ? 0 : side == 1 ? p : side == 2 ? HALO_W - 1 : HALO_W - 1 - p;
        const int gx = x0 - 1 + hx, gy = y0 - 1 + hy;
        int d = D_OUT;
        if (gx >= 0 && gy >= 0 && gx < R.W && gy < R.H) {
            const int c = (hy + 1) * ZW + hx + 1;
            float nb[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) nb[q] = U.zt[c + FDY[q] * ZW + FDX[q]];
            uint32_t dir;
            d = d8_of(U.zt[c], nb, gx, gy, R.W, R.H, dir);
        }
        T.d[hy * HALO_W + hx] = d;
    }
    // The tile, a column of its strip a thread, three rows of elevations in
    // registers.  Lane k keeps the words of the strip's row k.
    Row64 nbr[8], inf = 0, zero = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) nbr[q] = 0;
    {
        const float* col = U.zt + (strip * STRIP + 1) * ZW + lx + 1;
        float up[3], at[3], dn[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            up[j] = col[j];
            at[j] = col[ZW + j];
        }
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const int ly = strip * STRIP + k;
            const int gx = x0 + lx, gy = y0 + ly;
#pragma unroll
            for (int j = 0; j < 3; ++j) dn[j] = col[(k + 2) * ZW + j];
            const float nb[8] = {up[1], up[2], at[2], dn[2], dn[1], dn[0], at[0], up[0]};
            uint32_t dir;
            int d = d8_of(at[1], nb, gx, gy, R.W, R.H, dir);
            if (gx < R.W && gy < R.H)
                reinterpret_cast<uint16_t*>(R.fd)[(size_t)gy * R.W + gx] = (uint16_t)dir;
            else
                d = D_OUT;
            T.d[(ly + 1) * HALO_W + lx + 1] = d;
            const Row64 flat = __ballot(d == D_INF);
            row_write(inf, flat, k);
            row_write(zero, __ballot(d == 0), k);
            if (flat) {
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    row_write(nbr[q], flat & __ballot(nb[q] <= at[1]), k);
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                up[j] = at[j];
                at[j] = dn[j];
            }
        }
    }
    __syncthreads();  // every read of the elevations is done
    if (lx < STRIP) {
        const int r = strip * STRIP + lx;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            U.s.nbr[q][r] = nbr[q];
            fr_nbr(a, b, q)[r] = nbr[q];
        }
        T.inf[r] = inf;
        T.aux[r] = zero;
    }
    __syncthreads();
    Levels v;
    if (strip == 0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v.nbr[q] = U.s.nbr[q][lx];
    }
    const uint32_t changed = flat_solve(v, T, U.s.S, true);
    flat_finish(T, a, b, tx, ty, changed, true, a.work + (size_t)a.total, &a.ctrl[CTL_COUNT + 1],
                FR_EPOCH0);
}

// The flat passes, after k_fr_d8 (k_fr_pick follows).
// MULTI: a table of rasters (else the one raster of the arguments).
// Four waves a SIMD: the LDS of a flat tile allows four workgroups per CU.
template <bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_fr_persistent(FrArgs a) {
    __shared__ FrTile T;
    __shared__ FrSolve S;
    if (grid_aborted(a.gb)) return;
    uint32_t epoch = FR_EPOCH0;

    int li = 1;  // pass 0 ran in k_fr_d8 and filled list 1
    bool converged = false;
    int pass = 1;
    // after a pass the next list's count comes with the barrier (the sum of
    // what each workgroup listed) where the blocks are fewer than
    // BAR_SUM_LIMIT
    const bool sums = (uint64_t)a.total < BAR_SUM_LIMIT;
    uint32_t next_count = 0;
    for (; pass < a.max_passes; ++pass) {
        const int cin = li, cout = (li + 1) % 3, cclr = (li + 2) % 3;
        const uint32_t count = pass > 1 && sums ? next_count : ld(&a.ctrl[CTL_COUNT + cin]);
        if (count == 0) {
            converged = true;
            break;
        }
        ++epoch;
        if (blockIdx.x == 0 && threadIdx.x == 0) a.ctrl[CTL_COUNT + cclr] = 0;
        const int* win = a.work + (size_t)cin * a.total;
        int* wout = a.work + (size_t)cout * a.total;
        if (threadIdx.x == 0) T.pushed = 0u;
        for (uint32_t i = blockIdx.x; i < count; i += gridDim.x)
            bfs_tile(T, S, a, fr_block<MULTI>(a, win[i]), wout, &a.ctrl[CTL_COUNT + cout], epoch);
        uint32_t unused = 0;
        if (!grid_sync_sum(a.gb, 0, sums ? T.pushed : 0u, 0u, next_count, unused)) return;
        li = cout;
    }
    // The words written below are not read by the pass loop, so no barrier
    // is needed between the last count read and them.
    if (!converged) {
        if (blockIdx.x == 0 && threadIdx.x == 0)
            a.ctrl[CTL_STATUS] = (uint32_t)(-CAGEO_ERR_NOT_CONVERGED);
        return;
    }

    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.ctrl[CTL_FR_PASSES] = (uint32_t)pass;  // read by the host only
        a.ctrl[CTL_FR_DONE] = 1u;               // k_fr_pick may go on
    }
}

// Directions of the resolved flats (FlowRoutingAlgorithmCPUOpenMP.h:
// 153-249): the last neighbour in order with d(n) = d(c) - 1 and
// z_n <= z_c.  One workgroup per block: its own distances first (a block
// without a resolved flat is done), then the distances with a one-cell halo
// and the neighbour masks staged in LDS in one batch of loads; a halo cell
// outside the grid reads D_OUT, which no d(c) - 1 >= 0 equals.  Runs only
// after flat passes that converged (k_fr_persistent sets CTL_FR_DONE).
// Bound by its two rounds of loads; with the masks (a byte a cell) in place
// of the elevations 51 us at 4096^2, 71 before.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_fr_pick(FrArgs a) {
    __shared__ int d[FR_D];
    __shared__ Row64 nbr[8][TILE];
    if (ld(&a.ctrl[CTL_FR_DONE]) == 0u) return;
    const FrBlock b = fr_block<MULTI>(a, blockIdx.x);
    const FrRaster& R = b.R;
    const int x0 = (b.lb % R.ntx) * TILE, y0 = (b.lb / R.ntx) * TILE;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = x0 + lx;
    uint32_t flat = 0;
    {
        int32_t dv[STRIP];
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const int y = y0 + strip * STRIP + k;
            const bool in = x < R.W && y < R.H;
            dv[k] = R.dist[in ? (size_t)y * R.W + x : 0];
            if (!in) dv[k] = 0;
        }
#pragma unroll
        for (int k = 0; k < STRIP; ++k)
            if (dv[k] >= 1 && dv[k] < D_INF) flat |= 1u << k;
    }
    if (!__syncthreads_or(flat != 0u)) return;
    {
        constexpr int ITER = (FR_D + TILE_THREADS - 1) / TILE_THREADS;
        int v[ITER];
        Row64 m[2];
#pragma unroll
        for (int j = 0; j < ITER; ++j) {
            const int k = threadIdx.x + j * TILE_THREADS;
            const int hy = k / HALO_W, hx = k - hy * HALO_W;
            const int gx = x0 - 1 + hx, gy = y0 - 1 + hy;
            const bool in = k < FR_D && gx >= 0 && gy >= 0 && gx < R.W && gy < R.H;
            v[j] = R.dist[in ? (size_t)gy * R.W + gx : 0];
            if (!in) v[j] = D_OUT;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) m[j] = fr_nbr(a, b, 4 * j + strip)[lx];
#pragma unroll
        for (int j = 0; j < ITER; ++j) {
            const int k = threadIdx.x + j * TILE_THREADS;
            if (k < FR_D) d[k] = v[j];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) nbr[4 * j + strip][lx] = m[j];
    }
    __syncthreads();
    while (flat) {
        const int k = __builtin_ctz(flat);
        flat &= flat - 1;
        const int ly = strip * STRIP + k;
        const int li = (ly + 1) * HALO_W + lx + 1;
        const int want = d[li] - 1;
        bool found = false;
        char2 dir = make_char2(0, 0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (d[li + FDY[q] * HALO_W + FDX[q]] == want && ((nbr[q][ly] >> lx) & 1u)) {  // the last
                found = true;
                dir = make_char2((int8_t)FDX[q], (int8_t)FDY[q]);
            }
        }
        if (found) reinterpret_cast<char2*>(R.fd)[(size_t)(y0 + ly) * R.W + x] = dir;
    }
}

FrRaster fr_raster(Context* c, const float* z, int8_t* fd) {
    FrRaster R;
    R.z = z;
    R.fd = fd;
    R.dist = c->d_dist;
    R.nbr = reinterpret_cast<Row64*>(c->d_bent);
    R.W = c->W;
    R.H = c->H;
    R.ntx = c->ntx;
    R.nty = c->nty;
    return R;
}

}  // namespace

// Co-resident workgroups of the persistent kernel on this device.
int flow_routing_grid_cap(Context* c, int* cap) {
    int per_cu = 0;
    CAGEO_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void*>(k_fr_persistent<false>), TILE_THREADS, 0));
    hipDeviceProp_t prop;
    CAGEO_HIP_TRY(hipGetDeviceProperties(&prop, c->device));
    if (per_cu < 1) return CAGEO_ERR_HIP;
    *cap = per_cu * prop.multiProcessorCount;
    return CAGEO_OK;
}

int flow_routing(Context* c, const float* z, int8_t* fd) {
    if (c->fr_grid <= 0) CAGEO_TRY(flow_routing_grid_cap(c, &c->fr_grid));
    FrArgs a;
    a.one = fr_raster(c, z, fd);
    a.rs = nullptr;
    a.bmap = nullptr;
    a.total = c->ntiles;
    a.work = c->d_work3;
    a.mark = c->d_mark;
    a.nbr = reinterpret_cast<Row64*>(c->d_pfmask);
    a.ctrl = c->d_ctrl;
    a.gb = context_gridbar(c);
    a.max_passes = 1 << 20;
    hipLaunchKernelGGL(k_fr_reset, dim3((a.total + 255) / 256), dim3(256), 0, c->stream, a);
    hipLaunchKernelGGL(k_fr_d8<false>, dim3(a.total), dim3(TILE_THREADS), 0, c->stream, a);
    // ordinary launch within the occupancy cap (see pf_launch); no
    // more workgroups than blocks, as each adds to the barriers (the routing
    // of 1000 x 777, 208 blocks: 226 us, 277 with the full grid)
    hipLaunchKernelGGL(k_fr_persistent<false>, dim3(std::min(c->fr_grid, a.total)),
                       dim3(TILE_THREADS), 0, c->stream, a);
    hipLaunchKernelGGL(k_fr_pick<false>, dim3(a.total), dim3(TILE_THREADS), 0, c->stream, a);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

// Raster table of a batch: each context's d_w -> d_fd.
int flow_routing_tables(MultiState* m, Context* const* ctxs) {
    std::vector<FrRaster> t(m->nr);
    for (int r = 0; r < m->nr; ++r) t[r] = fr_raster(ctxs[r], ctxs[r]->d_w, ctxs[r]->d_fd);
    CAGEO_HIP_TRY(hipMalloc(&m->d_fr, t.size() * sizeof(FrRaster)));
    CAGEO_HIP_TRY(hipMemcpy(m->d_fr, t.data(), t.size() * sizeof(FrRaster), hipMemcpyHostToDevice));
    {
        int per_cu = 0;
        CAGEO_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void*>(k_fr_persistent<true>), TILE_THREADS, 0));
        hipDeviceProp_t prop;
        CAGEO_HIP_TRY(hipGetDeviceProperties(&prop, ctxs[0]->device));
        if (per_cu < 1) return CAGEO_ERR_HIP;
        m->fr_cap = per_cu * prop.multiProcessorCount;
    }
    if (m->fr_grid <= 0) m->fr_grid = m->fr_cap;
    return CAGEO_OK;
}

int flow_routing_multi(MultiState* m, hipStream_t s) {
    FrArgs a;
    a.one = FrRaster{};
    a.rs = static_cast<const FrRaster*>(m->d_fr);
    a.bmap = m->d_bmap;
    a.total = m->total;
    a.work = m->d_work;
    a.mark = m->d_mark_fr;
    a.nbr = reinterpret_cast<Row64*>(m->d_pfmask);
    a.ctrl = m->d_ctrl;
    a.gb = multi_gridbar(m);
    a.max_passes = 1 << 20;
    hipLaunchKernelGGL(k_fr_reset, dim3((a.total + 255) / 256), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_fr_d8<true>, dim3(a.total), dim3(TILE_THREADS), 0, s, a);
    hipLaunchKernelGGL(k_fr_persistent<true>, dim3(std::min(m->fr_grid, a.total)),
                       dim3(TILE_THREADS), 0, s, a);
    hipLaunchKernelGGL(k_fr_pick<true>, dim3(a.total), dim3(TILE_THREADS), 0, s, a);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

}  // namespace cageo
