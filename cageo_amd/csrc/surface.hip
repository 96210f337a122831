// Surface stages that turn the error field into the DEM the pit fill sees:
//  - RealisticDemAlgorithm<T,U>::execute, RealisticDemAlgorithm.h:49-70
//    (AddSurfacesAlgorithmCPUOpenMP.h:36-56 then
//    RemoveNegativeElevationsAlgorithmCPUOpenMP.h:34-48);
//  - StreamBurningAlgorithm<T,U>::execute, StreamBurningAlgorithm.h:116-134
//    with performStreamBurning, StreamBurningAlgorithmCPUOpenMP.h:32-82;
//  - the mm quantisation that opens performPitFilling,
//    PitFillingAlgorithmCPUOpenMP.h:84-106.
//
// Burning semantics.  The reference updates z in place while scanning each
// cell's circular search array; with one thread in raster order a stream
// neighbour n that precedes the cell has already been set to 0, one that
// follows still holds its realistic-DEM value.  Non-stream cell i takes
//   z_i * factor(o)  for the first offset o (order of
//                    StreamBurningAlgorithm.h:140-167) whose cell n is in the
//                    grid, is a stream cell, and has seen(n) != nodata_dem,
//                    seen(n) = n < i ? 0 : z_n;
//   z_i              otherwise;
// stream cells become 0.  Evaluated out of place here so every cell reads the
// unburned values.
#include <cmath>
#include <list>
#include <type_traits>
#include <vector>

#include "tiles.hpp"

namespace cageo {

namespace {


__global__ __launch_bounds__(256) void k_stream_flags(const float* __restrict__ stream,
                                                      int64_t n, float nodata_stream,
                                                      uint8_t* __restrict__ sflags,
                                                      int32_t* __restrict__ slabel) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        float s = stream[i];
        uint8_t f = 0;
        if (s != nodata_stream) f |= SF_BURN;  // StreamBurningAlgorithmCPUOpenMP.h:46
        if (s >= 0.0f) f |= SF_TRACE;          // FlowTracingAlgorithmCPUOpenMP.h:52,88
        sflags[i] = f;
        // FlowTracingAlgorithmCPUOpenMP.h:89: label = -stream converted to int
        slabel[i] = (s >= 0.0f) ? (int32_t)(-s) : 0;
    }
}

__device__ inline float realistic_value(float d, float e, float nodata) {
    float v = (d != nodata) ? d + e : e;
    if (v <= 0.0f && v != nodata) v = 1.0f;
    return v;
}

__global__ __launch_bounds__(256) void k_realistic(const float* __restrict__ dem,
                                                   float* __restrict__ field, int64_t n,
                                                   float nodata) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        field[i] = realistic_value(dem[i], field[i], nodata);
}

// Burning works on blocks of 64 x 32 cells, a wave for 8 rows of them.  What
// the search asks about a neighbour n is one of two facts, given that n is in
// the grid:
//   burn  n is a stream cell;
//   late  n is a stream cell whose unburned value is not nodata_dem.
// A neighbour that precedes the cell in raster order (offset dy < 0, or
// dy == 0 and dx < 0: for in-grid cells the reference's n < i reduces to
// the offset alone) has been burned to 0 already and qualifies when
// 0 != nodata_dem, i.e. by `burn` under that launch constant; a later one
// qualifies by `late`.  Both are kept as bit masks, a window of 64 + 2R cells
// a row (cells outside the grid have no bit, which is the reference's in-grid
// test): a cell's neighbourhood is then 2R + 1 bits of each of 2R + 1 words,
// and a distance's offsets are tested together, their factor being the same.
// Bound by its loads, all of them issued before the first is used.  A byte
// of flags a cell in LDS, read offset by offset, took 145 us at 4096^2 and
// 547 at 8192^2 (with the minimum and maximum); now 73 and 241 (a copy of as
// many bytes: 42 and 168).  Shifting uniform words offset by offset in scalar
// registers was slower, 169 and 613: a serial chain for each row.
constexpr int BT_X = 64, BT_R = 8, BT_Y = 4 * BT_R;
constexpr int BH_MAX = CAGEO_MAX_BEVEL_RADIUS;
constexpr int BE_Y = BT_Y + 2 * BH_MAX;  // rows of a block with its halo
static_assert(BH_MAX <= 8, "the 2R side cells of a row take 16 bits");
typedef unsigned long long Mask64;

// REAL: the tile's values are realistic_value(z0, z1) (the fused Monte
// Carlo pass), else z0 itself.  out[j]: burned value of column gx, row gy + j.
template <bool REAL, int R>
__device__ inline void burn_tile(int W, int H, const uint8_t* __restrict__ sf,
                                 const float* __restrict__ fac, int n_off, float nodata_dem,
                                 const float* __restrict__ z0, const float* __restrict__ z1,
                                 float out[BT_R], int& gx, int& gy) {
    constexpr int NH = (2 * R + 3) / 4;                          // halo rows of a wave
    constexpr int NS = R ? (16 * (BT_Y + 2 * R) + 255) / 256 : 0;  // side cells of a thread
    __shared__ Mask64 s_burn[BE_Y], s_late[BE_Y];  // the 64 cells of the block's columns
    __shared__ Mask64 s_sburn[NS * 4 + 1], s_slate[NS * 4 + 1];  // side cells, 16 bits a row
    // Blocks go round robin over the 8 XCDs; renumbering them so that each
    // XCD takes a contiguous band of tiles keeps the neighbours whose cache
    // lines hold this tile's halo in the same L2 (a bijection on the block
    // numbers when their count is a multiple of 8).
    const unsigned nb = gridDim.x * gridDim.y;
    unsigned t = blockIdx.y * gridDim.x + blockIdx.x;
    if ((nb & 7) == 0) t = (t & 7) * (nb >> 3) + (t >> 3);
    const int x0 = (int)(t % gridDim.x) * BT_X, y0 = (int)(t / gridDim.x) * BT_Y;
    const int lx = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    gx = x0 + lx;
    gy = y0 + wave * BT_R;
    // A cell outside the grid, or beyond the radius, loads cell 0 (cached)
    // and is replaced afterwards, so no load sits in a branch.
    struct Cell {
        float a, b;
        uint8_t f;
        bool in;
    };
    auto load = [&](int x, int y, bool want) {
        Cell c;
        c.in = want && x >= 0 && y >= 0 && x < W && y < H;
        const size_t i = c.in ? (size_t)y * W + x : 0;
        c.a = z0[i];
        c.b = REAL ? z1[i] : 0.0f;
        c.f = sf[i];
        return c;
    };
    Cell own[BT_R], halo[NH + 1], side[NS + 1];
#pragma unroll
    for (int j = 0; j < BT_R; ++j) own[j] = load(gx, gy + j, true);
#pragma unroll
    for (int j = 0; j < NH; ++j) {
        const int k = wave + 4 * j;  // halo row: R above, R below
        halo[j] = load(gx, k < R ? y0 - R + k : y0 + BT_Y + k - R, k < 2 * R);
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int i = threadIdx.x + 256 * j, c = i & 15, k = i >> 4;
        side[j] = load(c < R ? x0 - R + c : x0 + BT_X + c - R, y0 - R + k,
                       c < 2 * R && k < BT_Y + 2 * R);
    }
    auto value = [&](const Cell& c) { return REAL ? realistic_value(c.a, c.b, nodata_dem) : c.a; };
    auto masks = [&](const Cell& c, float v, Mask64& burn, Mask64& late) {
        const bool f = c.in && (c.f & SF_BURN);
        burn = __ballot(f);
        late = __ballot(f && v != nodata_dem);
    };
    Mask64 stream[BT_R];
#pragma unroll
    for (int j = 0; j < BT_R; ++j) {
        Mask64 late;
        out[j] = value(own[j]);
        masks(own[j], out[j], stream[j], late);
        s_burn[R + wave * BT_R + j] = stream[j];
        s_late[R + wave * BT_R + j] = late;
        if (own[j].f & SF_BURN) out[j] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NH; ++j) {
        const int k = wave + 4 * j;
        Mask64 burn, late;
        masks(halo[j], value(halo[j]), burn, late);
        if (k < 2 * R) {
            s_burn[k < R ? k : BT_Y + k] = burn;
            s_late[k < R ? k : BT_Y + k] = late;
        }
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        Mask64 burn, late;
        masks(side[j], value(side[j]), burn, late);
        s_sburn[4 * j + wave] = burn;
        s_slate[4 * j + wave] = late;
    }
    __syncthreads();
    if constexpr (R > 0) {
        // Row e of the wave's rows with their halo, as each lane sees it: bit
        // i is column gx + i - R.
        constexpr int E = BT_R + 2 * R, F = 2 * R + 1;
        uint32_t fb[E], fl[E];
        auto field = [&](Mask64 mid, uint32_t s) {
            const Mask64 lo = mid << R | (s & ((1u << R) - 1u));
            const Mask64 hi = mid >> (64 - R) | (Mask64)(s >> R) << R;
            return ((uint32_t)(lo >> lx) | (uint32_t)((hi << 1) << (63 - lx))) & ((1u << F) - 1u);
        };
        bool some = false;  // a stream cell in those rows
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int row = wave * BT_R + e;
            const uint32_t sb = (uint32_t)(s_sburn[row >> 2] >> (16 * (row & 3))) & 0xffffu;
            const uint32_t sl = (uint32_t)(s_slate[row >> 2] >> (16 * (row & 3))) & 0xffffu;
            fb[e] = nodata_dem != 0.0f ? field(s_burn[row], sb) : 0u;
            fl[e] = field(s_late[row], sl);
            some |= (fb[e] | fl[e]) != 0u;
        }
        if (!__any(some)) return;
#pragma unroll
        for (int j = 0; j < BT_R; ++j) {
            if (own[j].f & SF_BURN) continue;
            // Qualifying neighbours by row.  The search takes the first in
            // order of distance, and its factor depends on the distance only.
            uint32_t q[F];
#pragma unroll
            for (int d = 0; d < F; ++d) {
                const uint32_t before = (1u << R) - 1u;
                q[d] = d < R ? fb[j + d]
                             : d > R ? fl[j + d] : (fb[j + d] & before) | (fl[j + d] & ~before & ~(1u << R));
            }
            float f = 1.0f;
            int o = n_off;
            bool found = false;
#pragma unroll
            for (int d2 = R * R; d2 >= 1; --d2) {  // (the nearest is written last)
                int count = 0;
                uint32_t any = 0;
#pragma unroll
                for (int d = 0; d < F; ++d) {
                    uint32_t m = 0;
#pragma unroll
                    for (int i = 0; i < F; ++i)
                        if ((i - R) * (i - R) + (d - R) * (d - R) == d2) {
                            m |= 1u << i;
                            ++count;
                        }
                    any |= q[d] & m;
                }
                if (count == 0) continue;
                o -= count;
                if (any != 0) f = fac[o];
                found |= any != 0;
            }
            out[j] = found ? out[j] * f : out[j];
        }
    }
}

template <int R>
__global__ __launch_bounds__(256) void k_burn(const float* __restrict__ zin,
                                              float* __restrict__ zout,
                                              const uint8_t* __restrict__ sf,
                                              const float* __restrict__ fac, int n_off, int W, int H,
                                              float nodata_dem) {
    float v[BT_R];
    int gx, gy;
    burn_tile<false, R>(W, H, sf, fac, n_off, nodata_dem, zin, nullptr, v, gx, gy);
#pragma unroll
    for (int j = 0; j < BT_R; ++j)
        if (gx < W && gy + j < H) zout[(size_t)(gy + j) * W + gx] = v[j];
}

// Quantisation of PitFillingAlgorithmCPUOpenMP.h:84-106 for one value.
__device__ inline float quantize_mm(float v, float nodata, uint32_t* bad) {
    if (v == nodata) return v;
    if (v < 0.0f || v != v) {
        *bad = 1u;
        return v;
    }
    uint64_t q = pf_to_index(v, 0.0f);
    if (v != 0.0f && q == 0) q = 1;
    return pf_to_elev(q, 0.0f);
}

// (min, max) of ordered uints: "self after prev" of the wave scan.
__device__ inline void minmax_after(int& a, int& b, int pa, int pb) {
    a = (int)min((uint32_t)a, (uint32_t)pa);
    b = (int)max((uint32_t)b, (uint32_t)pb);
}

// Block-wide min/max of ordered uints (wave scans on DPP, then the four
// waves' results through LDS), then at most one atomic per word per block:
// a block whose value cannot improve the global word (which only moves
// one way) skips it, so the atomics do not queue on the three words.
__device__ inline void block_minmax(uint32_t mn, uint32_t mx, uint32_t bad, uint32_t* scal) {
    __shared__ uint32_t s_mn[4], s_mx[4], s_bad[4];
    int a = (int)mn, b = (int)mx;
    CAGEO_SCAN_UP(dpp_i, a, b, (int)0xffffffffu, 0, minmax_after);  // lane 63 holds the wave's
    const int w = threadIdx.x >> 6;
    const uint32_t wb = __any(bad != 0u) ? 1u : 0u;
    if ((threadIdx.x & 63) == 63) {
        s_mn[w] = (uint32_t)a;
        s_mx[w] = (uint32_t)b;
        s_bad[w] = wb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m0 = s_mn[0], m1 = s_mx[0], bb = s_bad[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
            m0 = min(m0, s_mn[k]);
            m1 = max(m1, s_mx[k]);
            bb |= s_bad[k];
        }
        if (m0 < __hip_atomic_load(&scal[SC_MIN], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&scal[SC_MIN], m0);
        if (m1 > __hip_atomic_load(&scal[SC_MAX], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&scal[SC_MAX], m1);
        if (bb) atomicOr(&scal[SC_BAD], bb);
    }
}

// The block's (min, max, bad) into part[0..2] (thread 0; plain stores, no
// wait on the global words): reduced by k_minmax_finish.
__device__ inline void block_minmax_store(uint32_t mn, uint32_t mx, uint32_t bad, uint32_t* part) {
    __shared__ uint32_t s_mn[4], s_mx[4], s_bad[4];
    int a = (int)mn, b = (int)mx;
    CAGEO_SCAN_UP(dpp_i, a, b, (int)0xffffffffu, 0, minmax_after);  // lane 63 holds the wave's
    const int w = threadIdx.x >> 6;
    const uint32_t wb = __any(bad != 0u) ? 1u : 0u;
    if ((threadIdx.x & 63) == 63) {
        s_mn[w] = (uint32_t)a;
        s_mx[w] = (uint32_t)b;
        s_bad[w] = wb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m0 = s_mn[0], m1 = s_mx[0], bb = s_bad[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
            m0 = min(m0, s_mn[k]);
            m1 = max(m1, s_mx[k]);
            bb |= s_bad[k];
        }
        part[0] = m0;
        part[1] = m1;
        part[2] = bb;
    }
}

// The raster's quantized min / max (ordered) and domain flag from the
// blocks' partials: one workgroup, its own loads of the partials all in
// flight per round, the three scalar words written once.
constexpr int MMF_T = 1024;
__global__ __launch_bounds__(MMF_T) void k_minmax_finish(const uint32_t* __restrict__ part, int nb,
                                                         uint32_t* __restrict__ scal) {
    uint32_t mn = 0xffffffffu, mx = 0u, bad = 0u;
#pragma unroll 8
    for (int i = threadIdx.x; i < nb; i += MMF_T) {
        mn = min(mn, part[3 * (size_t)i]);
        mx = max(mx, part[3 * (size_t)i + 1]);
        bad |= part[3 * (size_t)i + 2];
    }
    __shared__ uint32_t s_mn[MMF_T / 64], s_mx[MMF_T / 64], s_bad[MMF_T / 64];
    int a = (int)mn, b = (int)mx;
    CAGEO_SCAN_UP(dpp_i, a, b, (int)0xffffffffu, 0, minmax_after);
    const int w = threadIdx.x >> 6;
    const uint32_t wb = __any(bad != 0u) ? 1u : 0u;
    if ((threadIdx.x & 63) == 63) {
        s_mn[w] = (uint32_t)a;
        s_mx[w] = (uint32_t)b;
        s_bad[w] = wb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m0 = s_mn[0], m1 = s_mx[0], bb = s_bad[0];
        for (int k = 1; k < MMF_T / 64; ++k) {
            m0 = min(m0, s_mn[k]);
            m1 = max(m1, s_mx[k]);
            bb |= s_bad[k];
        }
        scal[SC_MIN] = m0;
        scal[SC_MAX] = m1;
        scal[SC_BAD] = bb;
    }
}

__global__ __launch_bounds__(256) void k_quantize_minmax(float* __restrict__ z, int64_t n,
                                                         float nodata,
                                                         uint32_t* __restrict__ scal) {
    uint32_t mn = 0xffffffffu, mx = 0u, bad = 0u;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        float q = quantize_mm(z[i], nodata, &bad);
        z[i] = q;
        uint32_t o = float_to_ordered(q);
        mn = min(mn, o);
        mx = max(mx, o);
    }
    block_minmax(mn, mx, bad, scal);
}

// Fused realistic DEM + burn + quantisation + min/max for the Monte Carlo
// driver: one pass over dem, error field and stream flags.  Each block
// leaves its min/max partial in `part` (3 words per block) for
// k_minmax_finish, so no block waits on the global words.
template <int R>
__global__ __launch_bounds__(256) void k_realistic_burn_quant(
    const float* __restrict__ dem, const float* __restrict__ e, const uint8_t* __restrict__ sf,
    const float* __restrict__ fac, int n_off, int W, int H, float nodata_dem, float* __restrict__ zq, uint32_t* __restrict__ part) {
    float v[BT_R];
    int gx, gy;
    burn_tile<true, R>(W, H, sf, fac, n_off, nodata_dem, dem, e, v, gx, gy);
    uint32_t mn = 0xffffffffu, mx = 0u, bad = 0u;
#pragma unroll
    for (int j = 0; j < BT_R; ++j) {
        if (gx < W && gy + j < H) {
            const float q = quantize_mm(v[j], nodata_dem, &bad);
            zq[(size_t)(gy + j) * W + gx] = q;
            const uint32_t o = float_to_ordered(q);
            mn = min(mn, o);
            mx = max(mx, o);
        }
    }
    block_minmax_store(mn, mx, bad, part + 3 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x));
}

// fn(a constant of the bevel radius): the radius is a template argument of
// the burning kernels.
template <class F>
int with_radius(int R, F fn) {
    static_assert(BH_MAX == 5, "every radius is listed");
    switch (R) {
        case 0: fn(std::integral_constant<int, 0>()); return CAGEO_OK;
        case 1: fn(std::integral_constant<int, 1>()); return CAGEO_OK;
        case 2: fn(std::integral_constant<int, 2>()); return CAGEO_OK;
        case 3: fn(std::integral_constant<int, 3>()); return CAGEO_OK;
        case 4: fn(std::integral_constant<int, 4>()); return CAGEO_OK;
        case 5: fn(std::integral_constant<int, 5>()); return CAGEO_OK;
        default: return CAGEO_ERR_ARG;
    }
}

inline unsigned grid_1d(size_t n) {
    size_t g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    return (unsigned)(g ? g : 1);
}

}  // namespace

// Circular search array of StreamBurningAlgorithm.h:140-167 ordered by
// (d^2, y, x) as coordDistCompare (StreamBurningCommon.cpp:13-28), with the
// bevel factor sqrt(d^2)/R of StreamBurningAlgorithmCPUOpenMP.h:67-71
// evaluated in float on the host.
int prepare_offsets(Context* c, int R) {
    if (R < 0 || R > CAGEO_MAX_BEVEL_RADIUS) return CAGEO_ERR_ARG;
    if (c->off_radius == R) return CAGEO_OK;
    struct O {
        int d, x, y;
    };
    std::list<O> l;
    for (int y = -R; y <= R; ++y)
        for (int x = -R; x <= R; ++x)
            if ((x || y) && x * x + y * y <= R * R) l.push_back({x * x + y * y, x, y});
    l.sort([](const O& a, const O& b) {
        return a.d < b.d || (a.d == b.d && (a.y < b.y || (a.y == b.y && a.x < b.x)));
    });
    std::vector<float> fac;
    for (const O& o : l) {
        float xd = (float)(-o.x), yd = (float)(-o.y);
        float dist = std::sqrt(xd * xd + yd * yd);
        fac.push_back(dist / (float)R);
    }
    c->n_offsets = (int)fac.size();
    if (c->n_offsets > 0) {
        CAGEO_HIP_TRY(hipMemcpyAsync(c->d_factor, fac.data(), fac.size() * sizeof(float),
                                     hipMemcpyHostToDevice, c->stream));
        CAGEO_HIP_TRY(hipStreamSynchronize(c->stream));
    }
    c->off_radius = R;
    return CAGEO_OK;
}

int launch_stream_flags(Context* c, const float* stream, float nodata_stream, uint8_t* sflags,
                        int32_t* slabel) {
    hipLaunchKernelGGL(k_stream_flags, dim3(grid_1d(c->n)), dim3(256), 0, c->stream, stream,
                       (int64_t)c->n, nodata_stream, sflags, slabel);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int launch_realistic(Context* c, const float* dem, float* field, float nodata) {
    hipLaunchKernelGGL(k_realistic, dim3(grid_1d(c->n)), dim3(256), 0, c->stream, dem, field,
                       (int64_t)c->n, nodata);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int launch_burn(Context* c, const float* zin, float* zout, const uint8_t* sflags,
                float nodata_dem) {
    dim3 grid((c->W + BT_X - 1) / BT_X, (c->H + BT_Y - 1) / BT_Y);
    CAGEO_TRY(with_radius(c->off_radius, [&](auto r) {
        hipLaunchKernelGGL(k_burn<r.value>, grid, dim3(256), 0, c->stream, zin, zout, sflags,
                           c->d_factor, c->n_offsets, c->W, c->H, nodata_dem);
    }));
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int launch_quantize(Context* c, float* dem, float nodata) {
    hipLaunchKernelGGL(k_quantize_minmax, dim3(grid_1d(c->n)), dim3(256), 0, c->stream, dem,
                       (int64_t)c->n, nodata, c->d_scal);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

// Blocks of k_realistic_burn_quant (the size of the context's d_bmm, 3 words each).
size_t burn_blocks(int W, int H) {
    return (size_t)((W + BT_X - 1) / BT_X) * (size_t)((H + BT_Y - 1) / BT_Y);
}

// Writes the raster's min / max / domain words (SC_MIN, SC_MAX, SC_BAD) as
// well: they need no reset before it.
int launch_realistic_burn_quant(Context* c, const float* dem, const float* e, float* zq) {
    dim3 grid((c->W + BT_X - 1) / BT_X, (c->H + BT_Y - 1) / BT_Y);
    CAGEO_TRY(with_radius(c->off_radius, [&](auto r) {
        hipLaunchKernelGGL(k_realistic_burn_quant<r.value>, grid, dim3(256), 0, c->stream, dem, e,
                           c->d_sflags, c->d_factor, c->n_offsets, c->W, c->H, c->nodata_dem, zq,
                           c->d_bmm);
    }));
    hipLaunchKernelGGL(k_minmax_finish, dim3(1), dim3(MMF_T), 0, c->stream, c->d_bmm,
                       (int)burn_blocks(c->W, c->H), c->d_scal);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

}  // namespace cageo
