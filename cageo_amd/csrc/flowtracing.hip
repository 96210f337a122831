// Flow tracing: FlowTracingAlgorithm<T,U,V>::execute, FlowTracingAlgorithm.h:
// 52-69; parity target FlowTracingAlgorithmCPUOpenMP.h:34-134.
//
// The reference walks every untraced cell along its directions until it
// leaves the grid (OUTSIDE), steps onto a stream cell (label = -stream as
// int) or onto an already labelled cell (copies it); stream cells themselves
// are LAKE; a walk longer than 100 001 steps (a cell with no direction, or a
// cycle) leaves its path at 0.  A cell's label is therefore the label of its
// path's terminal, computed here by pointer jumping in two levels:
//   1. per 64x64 tile, in LDS: every cell's pointer jumps along the in-tile
//      part of its path (12 doubling rounds cover 4096 cells) and ends at a
//      cell whose label is known, is "stuck" (its path cycles inside the
//      tile, e.g. a cell without a direction), or ends at a cell that exits
//      to another tile.  Cells of the first kind get their label at once, the
//      last keep the exit's slot and their steps to it as a positive code in
//      the label raster.  An exit lies on the tile's border and lands on a
//      border cell of the neighbouring tile, so the tile also writes the
//      entries of its own 252 border cells into a compact border table
//      (256 slots per tile);
//   2. over the border table only: exits jump through the entries of the
//      slots they name, in place, until no exit is left; a chain of more
//      steps than the raster has cells (or an entry holds), or of more hops
//      than there are slots, is a cycle through several tiles (stuck).  In place, and without
//      waiting for each other, is safe because every entry of a slot, old or
//      rewritten, names a slot on that cell's own path with the step count to
//      it, so a hop through either is correct, and a rewritten one is further
//      along;
//   3. every exit cell takes the label its tile's border slot resolved to.
// Table entries are 64 bits: kind (2 bits) | steps (30 bits) | value (32 bits), so
// the step count to the terminal is known and cells whose terminal is more
// than 100 001 steps away (where the reference's result depends on its
// raster order) are counted.  performConnectFlowPath (:115-134) then maps a
// label >= 0 (only 0 occurs: labels are -stream <= 0 or the negative
// constants) to label[0] when that is negative; it is applied in step 3.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "trace_steps.hpp"

namespace cageo {

namespace {

constexpr int BORDER_SLOTS = 256;

// Slot of tile cell (lx, ly) in its tile's border table: row 0 -> 0..63,
// row 63 -> 64..127, column 0 (rows 1..62) -> 129..190, column 63 (rows
// 1..62) -> 193..254; -1 inside.  Slots 128, 191, 192 and 255 stay unused.
__device__ inline int border_slot(int lx, int ly) {
    int s = -1;
    s = lx == TILE - 1 ? 3 * TILE + ly : s;
    s = lx == 0 ? 2 * TILE + ly : s;
    s = ly == TILE - 1 ? TILE + lx : s;
    return ly == 0 ? lx : s;
}

// Pointer of a cell within its tile: kind (2 bits) | steps (16 bits,
// saturated: a path of more than 4096 is a cycle) | LDS offset of a cell (14
// bits), K_LOCAL the cell its path has reached, else the cell where it ends.
constexpr uint32_t P_STEP1 = 1u << 14, P_STEPS = 0xffffu << 14, P_CELL = 0x3fffu;
__device__ inline uint32_t pointer(uint32_t kind, uint32_t steps, int cell) {
    return kind << 30 | steps << 14 | (uint32_t)cell << 2;
}
// Label of an exit cell between steps 1 and 3: a positive code, the cell it
// exits from and the steps to that cell (final labels are -stream ids, the
// negative constants, or 0).
__device__ inline int32_t exit_code(uint32_t p) { return (int32_t)(p & 0x3fffffffu) - (int32_t)P_STEP1 + 1; }
__device__ inline int exit_cell(int32_t code) { return ((code - 1) & (int32_t)P_CELL) >> 2; }
__device__ inline int exit_slot(int32_t code) {
    return border_slot(exit_cell(code) % TILE, exit_cell(code) / TILE);
}
__device__ inline uint32_t exit_steps(int32_t code) { return (uint32_t)(code - 1) / P_STEP1; }

// The tile pass of one tile.  A thread's 16 pointers stay in registers and
// the tile's in LDS (L), a word a cell.  Bound by its instructions, some 200
// a cell, and on a grid too small to fill the device by its three rounds of
// loads.  With 64-bit entries in LDS that carried the labels, read and
// tested one at a time, loads behind branches (each waited for by itself)
// and a 64-bit entry a cell for the exits in memory, the launch took 32 us
// at 1000 x 777 and 148 at 4096^2; now 12 and 68.
__device__ __forceinline__ void trace_tile(uint32_t* L, const int8_t* __restrict__ fd,
                                           const uint8_t* __restrict__ sf,
                                           const int32_t* __restrict__ slabel,
                                           int32_t* __restrict__ lab, uint64_t* __restrict__ bent,
                                           int W, int H, int ntx, int t) {
    const int tx = t % ntx, ty = t / ntx;
    const int x0 = tx * TILE, y0 = ty * TILE;
    const int lx = threadIdx.x & 63, strip = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gx = x0 + lx;
    const char2* dirs = reinterpret_cast<const char2*>(fd);

    // The strip's cells' flags and directions are loaded together, then
    // their targets' flags, then the labels of the targets on a stream.  No
    // load is conditional (one that is not wanted reads cell 0).  Cells are
    // numbered in 32 bits (a raster has fewer than 2^31).
    uint32_t e[STRIP];
    int32_t val[STRIP];  // of a cell where paths end: its label
    {
        const uint32_t first = (uint32_t)(y0 + strip * STRIP) * (uint32_t)W + (uint32_t)gx;
        const int rows = gx < W ? min(STRIP, H - (y0 + strip * STRIP)) : 0;
        uint8_t sfc[STRIP], sfn[STRIP];
        char2 dv[STRIP];
        uint32_t to[STRIP];
        uint32_t to_in = 0;  // cells in the grid whose target is
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const uint32_t i = k < rows ? first + (uint32_t)k * (uint32_t)W : 0u;
            sfc[k] = sf[i];
            dv[k] = dirs[i];
        }
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const int nx = gx + dv[k].x, ny = y0 + strip * STRIP + k + dv[k].y;
            const bool c = k < rows && (uint32_t)nx < (uint32_t)W && (uint32_t)ny < (uint32_t)H;
            to[k] = c ? (uint32_t)ny * (uint32_t)W + (uint32_t)nx : 0u;
            sfn[k] = sf[to[k]];
            to_in |= (uint32_t)c << k;
        }
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const bool c = ((to_in >> k) & 1u) && (sfn[k] & SF_TRACE);
            val[k] = slabel[c ? to[k] : 0u];
        }
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const int ly = strip * STRIP + k;
            const int li = ly * TILE + lx;
            const int dx = dv[k].x, dy = dv[k].y;
            const bool here = (uint32_t)(lx + dx) < (uint32_t)TILE && (uint32_t)(ly + dy) < (uint32_t)TILE;
            // the first that holds of: outside the grid, stream, off the
            // grid, onto a stream, no direction, in the tile, exit (a step
            // of more than one cell does not join borders: no path)
            uint32_t p = dx * dx + dy * dy <= 2 ? pointer(K_EXIT, 1, li) : pointer(K_STUCK, 0, li);
            p = here ? pointer(K_LOCAL, 1, li + dy * TILE + dx) : p;
            p = (dx | dy) == 0 ? pointer(K_STUCK, 0, li) : p;
            int32_t v = val[k];
            p = (sfn[k] & SF_TRACE) ? pointer(K_RESOLVED, 1, li) : p;
            const bool off = !((to_in >> k) & 1u);
            p = off ? pointer(K_RESOLVED, 1, li) : p;
            v = off ? CAGEO_FLOWTRACE_OUTSIDE : v;
            const bool lake = (sfc[k] & SF_TRACE) != 0;
            p = lake ? pointer(K_RESOLVED, 0, li) : p;
            v = lake ? CAGEO_FLOWTRACE_LAKE : v;
            p = k < rows ? p : pointer(K_STUCK, 0, li);
            e[k] = p;
            val[k] = v;
            L[li] = p;
        }
    }
    __syncthreads();
    const char* Lb = reinterpret_cast<const char*>(L);
    auto at = [&](uint32_t p) { return *reinterpret_cast<const uint32_t*>(Lb + (p & P_CELL)); };

    // Doubling rounds in place: a cell's pointer is written by its own
    // thread only, and the target's that it reads is either last round's or
    // already this round's, both exact summaries of the target's path.  So
    // every pointer at least doubles its hops a round (paths inside a tile
    // resolve within 13), step counts stay exact sums, and one barrier a
    // round suffices.
    for (int round = 0; round < 13; ++round) {
        uint32_t p[STRIP];
        uint32_t all = 0xffffffffu;
#pragma unroll
        for (int k = 0; k < STRIP; ++k) p[k] = at(e[k]);
#pragma unroll
        for (int k = 0; k < STRIP; ++k) {
            const uint32_t s = min((e[k] & P_STEPS) + (p[k] & P_STEPS), P_STEPS);
            const uint32_t n = (p[k] & ~P_STEPS) | s;
            e[k] = e[k] >> 30 == K_LOCAL ? n : e[k];
            L[(strip * STRIP + k) * TILE + lx] = e[k];
            all = min(all, e[k]);
        }
        static_assert(K_LOCAL == 0, "the least kind");
        if (!__syncthreads_or(all >> 30 == K_LOCAL)) break;
    }
    // The border cells, one a thread in the order of the slots: wave 0 the
    // first row, 1 the last, 2 the first column, 3 the last (rows 1 to 62;
    // the other four threads' slots are unused).
    const int bx = strip < 2 ? lx : strip == 2 ? 0 : TILE - 1;
    const int by = strip == 0 ? 0 : strip == 1 ? TILE - 1 : lx;
    const bool used = strip < 2 || (lx > 0 && lx < TILE - 1);
    const uint32_t bp = L[by * TILE + bx];
    int32_t slot = 0;  // that an exit leads to
    if (bp >> 30 == K_EXIT) {
        const int end = (int)((bp & P_CELL) >> 2);
        const uint32_t ex = (uint32_t)(x0 + end % TILE), ey = (uint32_t)(y0 + end / TILE);
        const char2 d = dirs[ey * (uint32_t)W + ex];
        const uint32_t nx = ex + (uint32_t)(int)d.x, ny = ey + (uint32_t)(int)d.y;
        slot = (int)((ny / TILE) * (uint32_t)ntx + nx / TILE) * BORDER_SLOTS +
               border_slot((int)(nx % TILE), (int)(ny % TILE));
    }
    __syncthreads();
    // Where paths end, the cell's label takes the pointer's place.
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const int li = (strip * STRIP + k) * TILE + lx;
        if ((e[k] & P_CELL) == (uint32_t)li << 2) L[li] = (uint32_t)val[k];
    }
    __syncthreads();
    // Outputs: labels and exit codes; the tile's border table, every slot
    // written (cells outside the grid and the four unused slots stuck).
    {
        const uint32_t kind = bp >> 30, steps = (bp & P_STEPS) / P_STEP1;
        uint64_t f = pack(K_STUCK, 0, 0);
        if (used && kind == K_RESOLVED) f = pack(K_RESOLVED, steps, (int32_t)at(bp));
        if (used && kind == K_EXIT) f = pack(K_EXIT, steps, slot);
        bent[(size_t)t * BORDER_SLOTS + threadIdx.x] = f;
    }
    int32_t* out = lab + (size_t)(y0 + strip * STRIP) * W + x0;
    const int rows = gx < W ? min(STRIP, H - (y0 + strip * STRIP)) : 0;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        const uint32_t kind = e[k] >> 30;
        int32_t label = (int32_t)at(e[k]);
        label = kind == K_RESOLVED ? label : 0;  // (K_LOCAL: a cycle inside the tile)
        label = kind == K_EXIT ? exit_code(e[k]) : label;
        if (k < rows) out[(size_t)k * W + lx] = label;
    }
}


__device__ inline uint32_t ld(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Entries read and rewritten by other waves during the exit rounds move as
// whole 64-bit words.
__device__ inline uint64_t ld64(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st64(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One raster of a launch.
struct TrRaster {
    const int8_t* fd;
    const uint8_t* sf;
    const int32_t* slabel;
    uint64_t* bent; // border table: BORDER_SLOTS entries per tile
    int32_t* lab;
    int W, H, ntx;
    uint32_t* scal;
};

// A launch over one raster (`one`, rs null) or over the rasters of a
// table, whose 64x64 blocks are numbered globally (bmap).
struct TrArgs {
    TrRaster one;
    const TrRaster* __restrict__ rs;
    const int2* __restrict__ bmap;  // per block: (raster, block within it)
    int total;
    uint32_t* ctrl;
    GridBar gb;     // status and abort words (no barrier is used)
};

struct TrBlock {
    TrRaster R;
    int lb;
};
template <bool MULTI>
__device__ inline TrBlock tr_block(const TrArgs& a, int g) {
    TrBlock b;
    g = __builtin_amdgcn_readfirstlane(g);
    if constexpr (!MULTI) {
        b.R = a.one;
        b.lb = g;
    } else {
        const int2 m = a.bmap[g];
        b.R = a.rs[__builtin_amdgcn_readfirstlane(m.x)];
        b.lb = __builtin_amdgcn_readfirstlane(m.y);
    }
    return b;
}

// Final label of cell 0 of a raster (between steps 2 and 3 of the launch).
__device__ inline int32_t label_of_cell0(const TrRaster& R) {
    const int32_t v = R.lab[0];
    if (v <= 0) return v;
    const uint64_t f = ld64(&R.bent[exit_slot(v)]);  // block 0's
    return kind_of(f) == K_RESOLVED ? value_of(f) : 0;
}

// Three launches over every raster: the tile pass (one workgroup per
// block), the border-table jumping and the exit cells' labels with the
// connect step (one workgroup per block).  All are light on registers, so
// many blocks' load chains are in flight at once, and none waits for
// another workgroup.

// Jumping rounds of the workgroups, by groups of them: the counters of the
// pit fill, idle here.
__device__ inline uint32_t* tr_rounds(const TrArgs& a, uint32_t group) {
    return a.ctrl + CTL_PF_COUNTS + group * CTL_PF_LINE;
}

// Tile pass.  Also clears the long-path and round counts: the launch
// boundary orders that before their first use.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_tr_tiles(TrArgs a) {
    __shared__ uint32_t L[TILE * TILE];
    const TrBlock b = tr_block<MULTI>(a, blockIdx.x);
    const TrRaster& R = b.R;
    if (b.lb == 0 && threadIdx.x == 0) R.scal[SC_LONGPATH] = 0;
    if (blockIdx.x == 0 && threadIdx.x < CTL_PF_GROUPS) *tr_rounds(a, threadIdx.x) = 0u;
    trace_tile(L, R.fd, R.sf, R.slabel, R.lab, R.bent, R.W, R.H, R.ntx, b.lb);
}

// Jumping over the border tables: thread s takes slot s % BORDER_SLOTS of
// global block s / BORDER_SLOTS (the blocks of one raster are consecutive,
// so a wave's 64 slots lie in one raster), and further ones a grid apart, a
// hop of each a round until none is an exit.  Threads run on without waiting
// for each other: a chain ends after at most as many hops as it has slots,
// whatever the others do, and the others' progress only shortens it.  The
// rounds are dependent loads at memory latency; with a grid barrier after
// each one the launch took 29 us at 1000 x 777 and 68 at 4096^2, now 5.5 and
// 11.5.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_tr_jump(TrArgs a) {
    if (grid_aborted(a.gb)) return;
    const long long slots = (long long)a.total * BORDER_SLOTS;
    uint32_t rounds = 0;
    for (bool pending = true; pending;) {
        ++rounds;
        pending = false;
        for (long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x; s < slots;
             s += (long long)gridDim.x * blockDim.x) {
            const TrBlock b = tr_block<MULTI>(a, (int)(s / BORDER_SLOTS));
            uint64_t* tb = b.R.bent;
            const size_t own = (size_t)b.lb * BORDER_SLOTS + (size_t)(s % BORDER_SLOTS);
            const uint64_t e = ld64(&tb[own]);
            if (kind_of(e) == K_EXIT) {
                uint64_t ne = hop(e, ld64(&tb[value_of(e)]));
                if (kind_of(ne) == K_EXIT) {
                    if (is_cycle(steps_of(ne), (uint32_t)b.R.W * (uint32_t)b.R.H) || rounds > slots)
                        ne = pack(K_STUCK, 0, 0);
                    else
                        pending = true;
                }
                st64(&tb[own], ne);
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) rounds = max(rounds, (uint32_t)__shfl_xor((int)rounds, off));
    if ((threadIdx.x & 63) == 0) atomicMax(tr_rounds(a, blockIdx.x % CTL_PF_GROUPS), rounds);
}

// Exit cells take their slot's label; performConnectFlowPath maps a label 0
// to label[0] when that is negative.  An exit whose chain is a cycle through
// tiles or ends stuck stays 0.  One workgroup per block, its border table in
// LDS, a wave per strip of STRIP rows (one lane per column).  One round of
// loads, where a 64-bit entry a cell and its slot's from another tile made
// it three: 23 us at 4096^2, 45 before.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_tr_exits(TrArgs a) {
    __shared__ uint64_t tb[BORDER_SLOTS];
    if (blockIdx.x == 0 && threadIdx.x < CTL_PF_GROUPS) {
        uint32_t r = ld(tr_rounds(a, threadIdx.x));
        for (int off = 32; off > 0; off >>= 1) r = max(r, (uint32_t)__shfl_xor((int)r, off));
        if (threadIdx.x == 0) a.ctrl[CTL_TR_ROUNDS] = r;  // read by the host only
    }
    const TrBlock b = tr_block<MULTI>(a, blockIdx.x);
    const TrRaster& R = b.R;
    const int x = (b.lb % R.ntx) * TILE + (threadIdx.x & 63);
    const int y0 = (b.lb / R.ntx) * TILE + (int)(threadIdx.x >> 6) * STRIP;
    const int rows = x < R.W ? min(STRIP, R.H - y0) : 0;
    static_assert(BORDER_SLOTS == TILE_THREADS, "a slot a thread");
    const uint64_t own = R.bent[(size_t)b.lb * BORDER_SLOTS + threadIdx.x];
    int32_t v[STRIP];
#pragma unroll
    for (int k = 0; k < STRIP; ++k) v[k] = k < rows ? R.lab[(size_t)(y0 + k) * R.W + x] : -1;
    const int32_t l0 = label_of_cell0(R);
    tb[threadIdx.x] = own;
    __syncthreads();
    uint32_t longp = 0;
#pragma unroll
    for (int k = 0; k < STRIP; ++k) {
        int32_t w = v[k];
        if (w > 0) {
            const uint64_t f = tb[exit_slot(w)];
            const uint32_t steps = exit_steps(w) + steps_of(f);
            w = 0;
            if (kind_of(f) == K_RESOLVED) {
                w = value_of(f);
                if (steps > 100001u) ++longp;  // past the walk guard
            }
        }
        if (w == 0 && l0 < 0) w = l0;
        if (w != v[k]) R.lab[(size_t)(y0 + k) * R.W + x] = w;
    }
    if (__any(longp)) {
        for (int off = 32; off > 0; off >>= 1) longp += (uint32_t)__shfl_xor((int)longp, off);
        if ((threadIdx.x & 63) == 0) {
            atomicAdd(&R.scal[SC_LONGPATH], longp);
            atomicAdd(&R.scal[SC_LONGRUN], longp);
        }
    }
}

// Workgroups of the jumping, as many as the device holds at once.
int jump_cap(const void* fn, int device, int* cap) {
    int per_cu = 0;
    CAGEO_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, TILE_THREADS, 0));
    hipDeviceProp_t prop;
    CAGEO_HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (per_cu < 1) return CAGEO_ERR_HIP;
    *cap = per_cu * prop.multiProcessorCount;
    return CAGEO_OK;
}

TrRaster tr_raster(Context* c, const int8_t* fd, const uint8_t* sflags, const int32_t* slabel,
                   int32_t* lab) {
    TrRaster R;
    R.fd = fd;
    R.sf = sflags;
    R.slabel = slabel;
    R.bent = c->d_bent;
    R.lab = lab;
    R.W = c->W;
    R.H = c->H;
    R.ntx = c->ntx;
    R.scal = c->d_scal;
    return R;
}

}  // namespace

// The long-path count is left in the scalar block.
int flow_tracing_grid_cap(Context* c, int* cap) {
    return jump_cap(reinterpret_cast<const void*>(k_tr_jump<false>), c->device, cap);
}

int flow_tracing(Context* c, const int8_t* fd, const uint8_t* sflags, const int32_t* slabel,
                 int32_t* lab, int64_t* long_paths) {
    if (c->tr_grid <= 0) CAGEO_TRY(flow_tracing_grid_cap(c, &c->tr_grid));
    TrArgs a;
    a.one = tr_raster(c, fd, sflags, slabel, lab);
    a.rs = nullptr;
    a.bmap = nullptr;
    a.total = c->ntiles;
    a.ctrl = c->d_ctrl;
    a.gb = context_gridbar(c);
    hipLaunchKernelGGL(k_tr_tiles<false>, dim3(a.total), dim3(TILE_THREADS), 0, c->stream, a);
    hipLaunchKernelGGL(k_tr_jump<false>, dim3(std::min(c->tr_grid, a.total)), dim3(TILE_THREADS), 0,
                       c->stream, a);
    hipLaunchKernelGGL(k_tr_exits<false>, dim3(a.total), dim3(TILE_THREADS), 0, c->stream, a);
    CAGEO_HIP_TRY(hipGetLastError());
    if (long_paths) {
        CAGEO_TRY(read_scalars(c));
        *long_paths = (int64_t)c->h_scal[SC_LONGPATH];
    }
    return CAGEO_OK;
}

// Raster table of a batch: each context's d_fd -> d_lab with its stream
// flags and labels.
int flow_tracing_tables(MultiState* m, Context* const* ctxs) {
    std::vector<TrRaster> t(m->nr);
    for (int r = 0; r < m->nr; ++r) {
        Context* c = ctxs[r];
        t[r] = tr_raster(c, c->d_fd, c->d_sflags, c->d_slabel, c->d_lab);
    }
    CAGEO_HIP_TRY(hipMalloc(&m->d_tr, t.size() * sizeof(TrRaster)));
    CAGEO_HIP_TRY(hipMemcpy(m->d_tr, t.data(), t.size() * sizeof(TrRaster), hipMemcpyHostToDevice));
    CAGEO_TRY(jump_cap(reinterpret_cast<const void*>(k_tr_jump<true>), ctxs[0]->device, &m->tr_cap));
    if (m->tr_grid <= 0) m->tr_grid = m->tr_cap;
    return CAGEO_OK;
}

int flow_tracing_multi(MultiState* m, hipStream_t s) {
    TrArgs a;
    a.one = TrRaster{};
    a.rs = static_cast<const TrRaster*>(m->d_tr);
    a.bmap = m->d_bmap;
    a.total = m->total;
    a.ctrl = m->d_ctrl;
    a.gb = multi_gridbar(m);
    hipLaunchKernelGGL(k_tr_tiles<true>, dim3(a.total), dim3(TILE_THREADS), 0, s, a);
    hipLaunchKernelGGL(k_tr_jump<true>, dim3(std::min(m->tr_grid, a.total)), dim3(TILE_THREADS), 0, s,
                       a);
    hipLaunchKernelGGL(k_tr_exits<true>, dim3(a.total), dim3(TILE_THREADS), 0, s, a);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

}  // namespace cageo
