// Kernels of the border-probability surrogate (a small U-Net): BF16 operands,
// FP32 accumulation on the MFMA units (v_mfma_f32_16x16x32_bf16), NHWC
// activations with channel counts that are multiples of 32.
//
// No reference counterpart: the reference has no learned part.  The network
// predicts the per-cell border frequency of the Monte Carlo from the DEM, the
// stream mask and the error model; the Monte Carlo generates its training
// maps and stays the judge of its output.
//
// 3x3 convolution as an implicit GEMM: rows = pixels, columns = output
// channels, K = 9 taps x input channels.  The input of a layer may be the
// concatenation of two tensors (decoder: upsampled deeper features and the
// skip connection), and the first of them may be read at half resolution
// (nearest upsampling folded into the load), so neither the concatenation
// nor the upsampled tensor is ever stored.
//
// MFMA operand layout (16x16x32, wave64): lane l holds 8 consecutive K values
// of row (l % 16) of A and of column (l % 16) of B, K block (l / 16); the
// accumulator holds rows 4*(l / 16) + r, r = 0..3, of column l % 16.
#include <type_traits>

#include "common.hpp"

namespace cageo {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t f2bf(float f) {  // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

struct ConvIn {
    const uint16_t* in1;  // [N][H1][W1][C1]; H1 = H/2, W1 = W/2 when up1
    const uint16_t* in2;  // [N][H][W][C2] or null
    int C1, C2, up1;
};

// 8 consecutive input channels [c, c+8) of pixel (n, y, x) of the (possibly
// concatenated, possibly upsampled) input; zero outside the image.
__device__ inline uint4 load_in8(const ConvIn& ci, int n, int y, int x, int H, int W, int c) {
    if (y < 0 || x < 0 || y >= H || x >= W) return make_uint4(0, 0, 0, 0);
    if (c < ci.C1) {
        const int H1 = ci.up1 ? (H + 1) / 2 : H, W1 = ci.up1 ? (W + 1) / 2 : W;
        const int yy = ci.up1 ? y / 2 : y, xx = ci.up1 ? x / 2 : x;
        return *reinterpret_cast<const uint4*>(ci.in1 + (((size_t)n * H1 + yy) * W1 + xx) * ci.C1 + c);
    }
    return *reinterpret_cast<const uint4*>(ci.in2 + (((size_t)n * H + y) * W + x) * ci.C2 + (c - ci.C1));
}

__device__ inline bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Forward 3x3 convolution (stride 1, zero padding 1).  One wave: 16*MT
// consecutive pixels x 16*NT output channels (MT x NT accumulator tiles, so
// each operand fragment loaded feeds NT or MT MFMAs); a workgroup of 4 waves
// covers 64*MT pixels.
// w: [9][Cout][Cin] bf16 (Cin = C1 + C2), bias: [Cout] fp32 or null.
// out: [N][H][W][Cout] bf16 (ReLU applied when relu), and/or outf fp32.
template <int NT, int MT>
__global__ __launch_bounds__(256) void k_conv3x3(ConvIn ci, const uint16_t* __restrict__ w,
                                                 const float* __restrict__ bias,
                                                 uint16_t* __restrict__ out,
                                                 float* __restrict__ outf, int N, int H, int W,
                                                 int Cout, int relu) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long M = (long long)N * H * W;
    const long long p0 = ((long long)blockIdx.x * 4 + wave) * 16 * MT;
    const int co0 = blockIdx.y * 16 * NT;
    if (p0 >= M) return;  // whole wave out of range (uniform)
    const int Cin = ci.C1 + ci.C2;
    const int row = lane & 15, kb = lane >> 4;
    int n[MT], y[MT], x[MT];
    bool pvalid[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const long long p = p0 + 16 * m + row;
        pvalid[m] = p < M;
        n[m] = y[m] = x[m] = 0;
        if (pvalid[m]) {
            n[m] = (int)(p / ((long long)H * W));
            const int r = (int)(p - (long long)n[m] * H * W);
            y[m] = r / W;
            x[m] = r - y[m] * W;
        }
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int tap = 0; tap < 9; ++tap) {
        const int dy = tap / 3 - 1, dx = tap % 3 - 1;
        const uint16_t* wt = w + (size_t)tap * Cout * Cin;
        for (int c = 0; c < Cin; c += 32) {
            const int cc = c + 8 * kb;
            bf16x8 a[MT], b[NT];
#pragma unroll
            for (int m = 0; m < MT; ++m)
                a[m] = as_bf16x8(pvalid[m] ? load_in8(ci, n[m], y[m] + dy, x[m] + dx, H, W, cc)
                                           : make_uint4(0, 0, 0, 0));
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int co = co0 + t * 16 + row;
                b[t] = as_bf16x8(*reinterpret_cast<const uint4*>(wt + (size_t)co * Cin + cc));
            }
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[t], acc[m][t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + t * 16 + row;  // accumulator column = lane % 16
        const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const long long pp = p0 + 16 * m + 4 * kb + r;  // accumulator row
                if (pp >= M) continue;
                float v = acc[m][t][r] + bv;
                if (relu) v = fmaxf(v, 0.0f);
                if (out) out[pp * Cout + co] = f2bf(v);
                if (outf) outf[pp * Cout + co] = v;
            }
    }
}

// The same convolution with its operands staged in LDS: for W % 64 == 0 and
// H % 4 == 0, and for any W and H where the input has one slice of 32 channels
// (EDGE: the tiles at the right and lower edges load zeros and store what
// lies inside).  A workgroup computes a tile of 4 rows x 64 pixels (a wave a
// row, 4 accumulator tiles of 16 pixels) x 16*NT output channels.  Per
// 32-channel slice of the input it stages the 6 x 66 input pixels the 9 taps
// read (zero outside the image, upsampling and concatenation folded into the
// loads) and the slice's weights of all 9 taps, then runs the 9 taps from LDS:
// each staged value is read from memory once per workgroup instead of once
// per tap and wave.
constexpr int CL_TX = 64;

// Place (in bf16) of 16-byte chunk c (0..3) of staged row r of the LDS
// convolution: a row is one pixel's (or one tap and output channel's) 32
// channels, 64 bytes with no padding, and its chunks are permuted by an XOR
// with bits 1-2 of the row number, so the rows a fragment read touches at
// once fall in distinct LDS banks.
__device__ inline int cl_at(int r, int c) { return r * 32 + 8 * (c ^ ((r >> 1) & 3)); }

struct ConvFuse {
    uint16_t* pool;       // [N][H/2][W/2][Cout]: k_avgpool2 of the output, or null
    const float* head_w;  // [Cout] and [1]: the 1x1 head of k_head
    const float* head_b;
    float* prob;          // [N][H][W] head output, or null (then head_w/head_b unused)
    int sigmoid;
    // a data gradient's ReLU backward: the output is masked by mask > 0
    // (bf16 [N][H][W][Cout]), and its sums over the pixels, the bias gradient
    // of the layer that made `mask`, go to dbias ([BIAS_SLOTS][Cout] partials)
    const uint16_t* mask;
    float* dbias;
};

// 0xffff halves where the bf16 halves of `a` are positive (a ReLU's output is
// never NaN).
__device__ inline uint32_t positive_halves(uint32_t a) {
    const uint32_t lo = (a & 0x8000u) == 0u && (a & 0x7fffu) != 0u ? 0xffffu : 0u;
    const uint32_t hi = (a & 0x80000000u) == 0u && (a & 0x7fff0000u) != 0u ? 0xffff0000u : 0u;
    return lo | hi;
}
__device__ inline uint4 relu_mask(uint4 v, uint4 a) {
    return make_uint4(v.x & positive_halves(a.x), v.y & positive_halves(a.y),
                      v.z & positive_halves(a.z), v.w & positive_halves(a.w));
}
// Adds 8 bf16 values to 8 sums.
__device__ inline void add8(float (&s)[8], uint4 v) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        s[2 * k] += bf2f((uint16_t)(u[k] & 0xffffu));
        s[2 * k + 1] += bf2f((uint16_t)(u[k] >> 16));
    }
}
// Sums over the workgroup (WAVES waves) of each thread's 8 channels
// 8 (threadIdx.x % CH) .. + 7, CH a power of two up to 32, added to this
// workgroup's slot of the partial sums: atomics of thousands of workgroups on
// one row of words would queue (23 ns each).  `part`: WAVES x 8 CH floats of
// LDS.
template <int WAVES = 4>
__device__ inline void bias_partials(float (&s)[8], int CH, float* part, float* dbias, int cout,
                                     int co0) {
    for (int off = 32; off >= CH; off >>= 1)
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] += __shfl_xor(s[k], off);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, C = 8 * CH;
    if (lane < CH)
#pragma unroll
        for (int k = 0; k < 8; ++k) part[wave * C + 8 * lane + k] = s[k];
    __syncthreads();
    if ((int)threadIdx.x < C) {
        float v = part[threadIdx.x];
        for (int k = 1; k < WAVES; ++k) v += part[k * C + threadIdx.x];
        atomicAdd(&dbias[(size_t)(blockIdx.x % BIAS_SLOTS) * cout + co0 + threadIdx.x], v);
    }
}

// What a workgroup of ROWS x CW waves makes of its accumulators: wave k's are
// row k % ROWS of the tile of ROWS rows x 64 pixels and output channels
// 16 NT (k / ROWS) on.  `smem` holds conv_out_words words that no wave uses
// any more.
//
// Without an fp32 output the results go out through LDS: the workgroup's
// bias + ReLU outputs, rounded to bf16, are staged there, then written
// with 16-byte stores (a pixel's channels are contiguous), and the fused
// consumers of the output read them there (ConvFuse): the 2x2 average pool
// and the 1x1 head, each in the same arithmetic as its own kernel
// (k_avgpool2, k_head), so a fused layer gives the same bits as the layer
// followed by that kernel.
template <int NT, int ROWS, int CW>
constexpr int conv_out_words() {
    constexpr int CO = 16 * NT * CW, NPX = ROWS * CL_TX;
    return NPX * (CO + 8) > CO * (NPX + 2) ? NPX * (CO + 8) : CO * (NPX + 2);
}
template <int NT, int ROWS, int CW, bool EDGE>
__device__ __forceinline__ void conv_out(f32x4 (&acc)[4][NT], uint16_t* smem,
                                         const float* __restrict__ bias, uint16_t* __restrict__ out,
                                         float* __restrict__ outf, const ConvFuse& fz, int n, int y0,
                                         int x0, int co0, int H, int W, int Cout, int relu) {
    constexpr int T = 64 * ROWS * CW, CO = 16 * NT * CW;
    constexpr int NPX = ROWS * CL_TX;    // pixels of the output tile
    constexpr int PS = CO + 8;           // staged pixel stride (bf16), padded by 16 bytes
    constexpr int HP = NPX + 2;          // staged channel stride of the head's layout
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kb = lane >> 4;
    const int wr = wave % ROWS, wc = 16 * NT * (wave / ROWS);
    if (outf) {  // fp32 output too: straight from the accumulators
        const long long prow = ((long long)n * H + y0 + wr) * W + x0;
        const int wx = W - x0;  // the tile's pixels inside
        if (EDGE && y0 + wr >= H) return;
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int co = co0 + wc + 16 * q + row;  // accumulator column = lane % 16
            const float bias_co = bias ? bias[co] : 0.0f;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (EDGE && 16 * m + 4 * kb + r >= wx) continue;
                    const long long pp = prow + 16 * m + 4 * kb + r;
                    float v = acc[m][q][r] + bias_co;
                    if (relu) v = fmaxf(v, 0.0f);
                    if (out) out[pp * Cout + co] = f2bf(v);
                    outf[pp * Cout + co] = v;
                }
        }
        return;
    }
    // the output tile's pixel (0, 0) in the NHWC raster; the head layout is
    // channel-major (a thread then reads its pixel's channels in order, lanes
    // on consecutive pixels), the other pixel-major
    const size_t pix0 = ((size_t)n * H + y0) * W + x0;
    const bool head = fz.prob != nullptr;
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int c = wc + 16 * q + row;  // accumulator column = lane % 16
        const float bias_co = bias ? bias[co0 + c] : 0.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int px = wr * CL_TX + 16 * m + 4 * kb + r;
                float v = acc[m][q][r] + bias_co;
                if (relu) v = fmaxf(v, 0.0f);
                smem[head ? c * HP + px : px * PS + c] = f2bf(v);
            }
    }
    __syncthreads();
    if (head) {  // CO == Cout (the host checks): the workgroup holds every channel
        for (int px = threadIdx.x; px < NPX; px += T) {
            if (EDGE && (px / CL_TX >= H - y0 || px % CL_TX >= W - x0)) continue;
            float s = fz.head_b[0];
            for (int c = 0; c < CO; ++c) s += fz.head_w[c] * bf2f(smem[c * HP + px]);
            fz.prob[pix0 + (size_t)(px / CL_TX) * W + px % CL_TX] =
                fz.sigmoid ? 1.0f / (1.0f + expf(-s)) : s;
        }
        return;
    }
    constexpr int CH = CO / 8;  // 16-byte chunks of a pixel's channels
    if (fz.mask) {
        float sum[8] = {};
#pragma unroll
        for (int i0 = 0; i0 < NPX * CH; i0 += T) {
            const int i = i0 + threadIdx.x, px = i / CH, part = i - px * CH;
            if (EDGE && (px / CL_TX >= H - y0 || px % CL_TX >= W - x0)) continue;
            const size_t o = (pix0 + (size_t)(px / CL_TX) * W + px % CL_TX) * Cout + co0 + 8 * part;
            const uint4 v = relu_mask(*reinterpret_cast<const uint4*>(smem + px * PS + 8 * part),
                                      *reinterpret_cast<const uint4*>(fz.mask + o));
            *reinterpret_cast<uint4*>(out + o) = v;
            add8(sum, v);
        }
        __syncthreads();  // the staged outputs are read
        bias_partials<ROWS * CW>(sum, CH, reinterpret_cast<float*>(smem), fz.dbias, Cout, co0);
        return;
    }
    if (out) {
        for (int i = threadIdx.x; i < NPX * CH; i += T) {
            const int px = i / CH, part = i - px * CH;
            if (EDGE && (px / CL_TX >= H - y0 || px % CL_TX >= W - x0)) continue;
            const size_t g = (pix0 + (size_t)(px / CL_TX) * W + px % CL_TX) * Cout + co0 + 8 * part;
            *reinterpret_cast<uint4*>(out + g) =
                *reinterpret_cast<const uint4*>(smem + px * PS + 8 * part);
        }
    }
    if (ROWS > 1 && fz.pool) {
        const int Wo = W / 2;
        const size_t q0 = ((size_t)n * (H / 2) + y0 / 2) * Wo + x0 / 2;
        for (int i = threadIdx.x; i < NPX / 4 * CH; i += T) {
            const int pp = i / CH, part = i - pp * CH;
            const int py = pp / (CL_TX / 2), px = pp - py * (CL_TX / 2);
            if (EDGE && (2 * py >= H - y0 || 2 * px >= W - x0)) continue;
            const uint16_t* s00 = smem + (2 * py * CL_TX + 2 * px) * PS + 8 * part;
            const uint4 a = *reinterpret_cast<const uint4*>(s00);                 // (2y, 2x)
            const uint4 b = *reinterpret_cast<const uint4*>(s00 + PS);            // (2y, 2x+1)
            const uint4 c = *reinterpret_cast<const uint4*>(s00 + CL_TX * PS);    // (2y+1, 2x)
            const uint4 d = *reinterpret_cast<const uint4*>(s00 + (CL_TX + 1) * PS);
            const uint32_t ua[4] = {a.x, a.y, a.z, a.w}, ub[4] = {b.x, b.y, b.z, b.w};
            const uint32_t uc[4] = {c.x, c.y, c.z, c.w}, ud[4] = {d.x, d.y, d.z, d.w};
            uint32_t res[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t h2 = 0;
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const int sh = 16 * hh;
                    const float sum = bf2f((uint16_t)(ua[k] >> sh)) + bf2f((uint16_t)(ub[k] >> sh)) +
                                      bf2f((uint16_t)(uc[k] >> sh)) + bf2f((uint16_t)(ud[k] >> sh));
                    h2 |= (uint32_t)f2bf(0.25f * sum) << sh;
                }
                res[k] = h2;
            }
            *reinterpret_cast<uint4*>(fz.pool + (q0 + (size_t)py * Wo + px) * Cout + co0 + 8 * part) =
                make_uint4(res[0], res[1], res[2], res[3]);
        }
    }
}

// EDGE: W or H is no multiple of the tile's (else the stores need no tests:
// with them a 4096^2 prediction takes 2 % longer).
template <int NT, int WPE, bool EDGE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void k_conv3x3_lds(ConvIn ci, const uint16_t* __restrict__ w,
                                                     const float* __restrict__ bias,
                                                     uint16_t* __restrict__ out,
                                                     float* __restrict__ outf, ConvFuse fz,
                                                     int N, int H, int W, int Cout, int relu) {
    constexpr int TY = 4, AX = CL_TX + 2, AY = TY + 2, CO = 16 * NT;
    constexpr int SA_N = AY * AX * 32, SB_N = 9 * CO * 32;
    static_assert(conv_out_words<NT, 4, 1>() <= SA_N + SB_N, "epilogue staging");
    __shared__ __align__(16) uint16_t smem[SA_N + SB_N];
    uint16_t* const sa = smem;
    uint16_t* const sb = smem + SA_N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kb = lane >> 4;
    const int tiles_x = EDGE ? (W + CL_TX - 1) / CL_TX : W / CL_TX;
    const int tiles_y = EDGE ? (H + TY - 1) / TY : H / TY;
    const int t = blockIdx.x;
    const int n = t / (tiles_x * tiles_y);
    const int ty = (t / tiles_x) % tiles_y, tx = t % tiles_x;
    const int x0 = tx * CL_TX, y0 = ty * TY;
    const int co0 = blockIdx.y * CO;
    const int Cin = ci.C1 + ci.C2;
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[m][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Slice c's loads are issued before slice c - 32's MFMAs and stored to
    // LDS after them, so their latency hides behind the arithmetic.  Input
    // AY x AX pixels x 4 groups of 8 channels, weights 9 taps x CO output
    // channels x 4 groups of 8 input channels.  What does not depend on the
    // slice is worked out once: each staged input value's pixel in in1 (at
    // half resolution with up1) and in in2, -1 outside the image, and each
    // weight value's offset.  A slice lies in one of the two inputs (their
    // channel counts are multiples of 32).
    constexpr int AN = AY * AX * 4, AIT = (AN + 255) / 256;
    constexpr int BN = 9 * CO * 4, BIT = (BN + 255) / 256;
    const int H1 = ci.up1 ? (H + 1) / 2 : H, W1 = ci.up1 ? (W + 1) / 2 : W;
    int pix1[AIT], pix2[AIT], boff[BIT];
#pragma unroll
    for (int j = 0; j < AIT; ++j) {
        const int i = threadIdx.x + 256 * j;
        const int px = i >> 2, yy = y0 - 1 + px / AX, xx = x0 - 1 + px % AX;
        const bool in = i < AN && yy >= 0 && xx >= 0 && yy < H && xx < W;
        pix1[j] = in ? (n * H1 + (ci.up1 ? yy / 2 : yy)) * W1 + (ci.up1 ? xx / 2 : xx) : -1;
        pix2[j] = in ? (n * H + yy) * W + xx : -1;
    }
#pragma unroll
    for (int j = 0; j < BIT; ++j) {
        const int i = threadIdx.x + 256 * j, r = i >> 2;  // r = tap * CO + co
        const int tap = r / CO, co = r - tap * CO;
        boff[j] = i < BN ? (tap * Cout + co0 + co) * Cin + 8 * (i & 3) : -1;
    }
    uint4 av[AIT], bv[BIT];
    auto load_slice = [&](int c) {
        const bool first = c < ci.C1;
        const uint16_t* src = first ? ci.in1 : ci.in2;
        const int cs = first ? ci.C1 : ci.C2, c0 = (first ? c : c - ci.C1) + 8 * (threadIdx.x & 3);
#pragma unroll
        for (int j = 0; j < AIT; ++j) {
            const int px = first ? pix1[j] : pix2[j];
            av[j] = px >= 0 ? *reinterpret_cast<const uint4*>(src + (size_t)px * cs + c0)
                            : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int j = 0; j < BIT; ++j)
            bv[j] = boff[j] >= 0 ? *reinterpret_cast<const uint4*>(w + boff[j] + c)
                                 : make_uint4(0u, 0u, 0u, 0u);
    };
    load_slice(0);
    for (int c = 0; c < Cin; c += 32) {
        __syncthreads();  // the last slice's reads are done
#pragma unroll
        for (int j = 0; j < AIT; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < AN) *reinterpret_cast<uint4*>(&sa[cl_at(i >> 2, i & 3)]) = av[j];
        }
#pragma unroll
        for (int j = 0; j < BIT; ++j) {
            const int i = threadIdx.x + 256 * j;
            if (i < BN) *reinterpret_cast<uint4*>(&sb[cl_at(i >> 2, i & 3)]) = bv[j];
        }
        __syncthreads();
        if (c + 32 < Cin) load_slice(c + 32);
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int dy = tap / 3, dx = tap % 3;  // halo-shifted offsets 0..2
            bf16x8 a[4], b[NT];
#pragma unroll
            for (int m = 0; m < 4; ++m)
                a[m] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &sa[cl_at((wave + dy) * AX + 16 * m + row + dx, kb)]));
#pragma unroll
            for (int q = 0; q < NT; ++q)
                b[q] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &sb[cl_at(tap * CO + 16 * q + row, kb)]));
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 0; q < NT; ++q)
                    acc[m][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[q], acc[m][q], 0, 0, 0);
        }
    }
    __syncthreads();  // every wave's operand reads of the last slice are done
    conv_out<NT, 4, 1, EDGE>(acc, smem, bias, out, outf, fz, n, y0, x0, co0, H, W, Cout, relu);
}

// The convolution for any W and H with its sums in k_conv3x3's order, all
// channels of tap 0 first, then those of tap 1, and so on (k_conv3x3_lds goes
// slice by slice), so that an image's outputs have the same bits whichever of
// the two kernels its size goes to.  The order needs every channel of the
// pixels at hand: a workgroup stages all of them once, in slices of 32 (see
// cl_at), an upsampled input at its own resolution, and then runs the steps,
// a slice of a tap each, with a step's weights through LDS.  While step j's
// products run, step j + 1's operands come from LDS, the weights of j + 2 go
// there and those of the three after it are on their way from memory.
// ROWS rows x 64 pixels a workgroup, ROWS x CW waves, each a row and 16 NT
// output channels.
// Bound by the LDS reads of a step (384 cycles for 256 of products with eight
// waves) and their latency; a barrier every three steps instead of one each
// gained 1 %.  The pixels often take the LDS of one workgroup a CU, so eight
// waves are better than four that reuse more (384 -> 128 channels upsampled
// at 252 x 176: 82 us against 101; with the upsampled input staged at full
// size, which leaves room for one row, 186).  A 1001 x 700 prediction takes
// 0.52 ms; with k_conv3x3 in its place 1.18, with the staged kernel's order
// 0.44.
constexpr int CT_LDS = 160 * 1024;
// Staged pixels of an input: whole eights, so that cl_at of a slice's pixel is
// the slice's place plus the pixel's.
constexpr int CT_AX = CL_TX + 2, CT_HX = CL_TX / 2 + 2;  // a row of them; of an upsampled input's
constexpr int conv_taps_px(int rows, int up) {
    return (up ? (rows / 2 + 2) * CT_HX + 7 : (rows + 2) * CT_AX + 7) & ~7;
}
// Words of LDS: the pixels, 8 that are written for none, two steps' weights.
constexpr int conv_taps_words(int rows, int block, int c1, int up1, int c2) {
    return conv_taps_px(rows, up1) * c1 + conv_taps_px(rows, 0) * c2 + 8 + 2 * 32 * block;
}
template <int NT, int ROWS, int CW>
__global__ __launch_bounds__(64 * ROWS * CW) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_conv3x3_taps(
    ConvIn ci, const uint16_t* __restrict__ w, const float* __restrict__ bias,
    uint16_t* __restrict__ out, float* __restrict__ outf, ConvFuse fz, int N, int H, int W, int Cout,
    int relu) {
    extern __shared__ __align__(16) uint16_t staged[];  // [slices][pixels][32], weights [2][CO][32]
    constexpr int T = 64 * ROWS * CW, CO = 16 * NT * CW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kb = lane >> 4;
    const int tiles_x = (W + CL_TX - 1) / CL_TX, tiles_y = (H + ROWS - 1) / ROWS;
    const int t = blockIdx.x;
    const int n = t / (tiles_x * tiles_y);
    const int y0 = (t / tiles_x) % tiles_y * ROWS, x0 = t % tiles_x * CL_TX;
    const int co0 = blockIdx.y * CO;
    const int Cin = ci.C1 + ci.C2;
    const int np1 = conv_taps_px(ROWS, ci.up1), np2 = conv_taps_px(ROWS, 0);
    const int words = np1 * ci.C1 + np2 * ci.C2;
    // Pixels of an input of Hs x Ws from (ys, xs) on, AX a row, to staged
    // pixel `r0` on: 16 bytes a load, a pixel's channels and then the next
    // pixel's by consecutive threads, B loads a thread under way (a pixel
    // outside loads the first one).
    auto stage = [&](auto row_of, const uint16_t* src, int C, int np, int Hs, int Ws, int ys, int xs,
                     int r0) __attribute__((always_inline)) {
        constexpr int B = 8, AX = row_of.value;
        const int cq = C / 8, dp = T / cq, dq = T - dp * cq;
        int p = threadIdx.x / cq, q = threadIdx.x - p * cq;
        while (__any(p < np)) {
            bf16x8 v[B];
            int at[B];
            uint32_t in = 0;
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const int py = p / AX, yy = ys + py, xx = xs + p - py * AX;
                const bool inside = p < np && yy >= 0 && xx >= 0 && yy < Hs && xx < Ws;
                const size_t o = (((size_t)n * Hs + yy) * Ws + xx) * C + 8 * q;
                v[k] = *reinterpret_cast<const bf16x8*>(src + (inside ? o : 0));
                in |= inside ? 1u << k : 0u;
                at[k] = p < np ? cl_at(r0 + (q >> 2) * np + p, q & 3) : words;
                p += dp;
                q += dq;
                if (q >= cq) {
                    q -= cq;
                    ++p;
                }
            }
#pragma unroll
            for (int k = 0; k < B; ++k)
                *reinterpret_cast<bf16x8*>(&staged[at[k]]) = (in >> k) & 1u ? v[k] : bf16x8{};
        }
    };
    constexpr int D = 3;        // steps a round: 9 taps make whole rounds of them
    constexpr int WT = CO * 4;  // threads with weights to stage
    static_assert(WT <= T, "a load a thread");
    bf16x8 a[D][4], b[D][NT], wv[D];
    // Weights: of the step to load (past the last, step 0's), this thread's
    // place in them, and where they go.
    const int wt = min((int)threadIdx.x, WT - 1);
    const uint32_t wlane = (uint32_t)((co0 + (wt >> 2)) * Cin + 8 * (wt & 3));
    const int wput = words + 8 + cl_at(wt >> 2, wt & 3);
    int ltap = 0, lc = 0;
    const uint16_t* wl = w;
    auto load = [&](bf16x8& v) __attribute__((always_inline)) {
        v = *reinterpret_cast<const bf16x8*>(wl + wlane);
        lc += 32;
        wl += 32;
        if (lc == Cin) {
            lc = 0;
            wl += (size_t)(Cout - 1) * Cin;
            if (++ltap == 9) {
                ltap = 0;
                wl = w;
            }
        }
    };
    auto put = [&](int slot, bf16x8 v) __attribute__((always_inline)) {
        if (WT == T || wave < WT / 64)
            *reinterpret_cast<bf16x8*>(&staged[wput + slot * CO * 32]) = v;
    };
    // Operands of the next step: its tap and slice (first staged pixel, first
    // channel), and where the tap's first pixel lies in a slice of either input.
    const int wread = words + 8 + cl_at(16 * NT * (wave / ROWS) + row, kb);
    int tap = 0, base = 0, c = 0, full = 0, half = 0;
    auto place = [&]() __attribute__((always_inline)) {
        const int y = wave % ROWS + tap / 3, x = row + tap % 3;
        full = cl_at(y * CT_AX + x, kb);
        half = cl_at(((y + 1) >> 1) * CT_HX + ((x + 1) >> 1), kb);
    };
    place();
    auto read = [&](int slot, bf16x8 (&a)[4], bf16x8 (&b)[NT]) __attribute__((always_inline)) {
        const bool first = c < ci.C1, up = first && ci.up1;
        const int at = (up ? half : full) + base * 32, step = up ? 8 * 32 : 16 * 32;
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = *reinterpret_cast<const bf16x8*>(&staged[at + m * step]);
#pragma unroll
        for (int q = 0; q < NT; ++q)
            b[q] = *reinterpret_cast<const bf16x8*>(&staged[wread + slot * CO * 32 + 16 * q * 32]);
        base += first ? np1 : np2;
        c += 32;
        if (c == Cin) {
            c = base = 0;
            tap = tap < 8 ? tap + 1 : 0;
            place();
        }
    };
    load(wv[0]);
    load(wv[1]);
    if (ci.up1)
        stage(std::integral_constant<int, CT_HX>(), ci.in1, ci.C1, np1, H / 2, W / 2, y0 / 2 - 1,
              x0 / 2 - 1, 0);
    else
        stage(std::integral_constant<int, CT_AX>(), ci.in1, ci.C1, np1, H, W, y0 - 1, x0 - 1, 0);
    if (ci.C2)
        stage(std::integral_constant<int, CT_AX>(), ci.in2, ci.C2, np2, H, W, y0 - 1, x0 - 1,
              np1 * (ci.C1 / 32));
    put(0, wv[0]);
    put(1, wv[1]);
    load(wv[2]);
    load(wv[0]);
    load(wv[1]);
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[m][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    read(0, a[0], b[0]);
    int slot = 0;  // of the step
    for (int s = 0; s < 9 * Cin; s += 32 * D) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            __syncthreads();  // step j + 1's weights are there, j's read
            // (left to itself the scheduler moves the loads down to their use)
            read(slot ^ 1, a[(j + 1) % D], b[(j + 1) % D]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 0; q < NT; ++q)
                    acc[m][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][m], b[j][q], acc[m][q], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            put(slot, wv[(j + 2) % D]);
            load(wv[(j + 2) % D]);
            slot ^= 1;
        }
    }
    __syncthreads();  // every wave's operand reads are done
    conv_out<NT, ROWS, CW, true>(acc, staged, bias, out, outf, fz, n, y0, x0, co0, H, W, Cout, relu);
}

// Weight gradient of the 3x3 convolution:
//   dW[tap][co][ci] += sum_p g[p][co] * x[p shifted by tap][ci]
// (GEMM rows co, columns ci, K = pixels).  A workgroup of 8 waves takes CO
// output x 32 input channels, all nine taps, over a 64-pixel wide run of image
// rows, two rows of g a step.
//
// Both operands want their channel's pixels in a row (K), but the rasters
// have a pixel's channels in a row: what is loaded (4 pixels x 8 channels a
// thread, 16-byte loads) is transposed in registers by byte permutes and
// stored to LDS channel-major, once for the nine taps.  The row taps are
// other rows of a ring of six x rows; the column taps are the same 8 pixels
// shifted by one, made from a fragment and the pixel pairs beside it by five
// bit alignments.  So a wave's K chunk of 32 pixels takes 2 fragments of g
// and, per row tap, one of x and two pairs, for 18 MFMAs.
//
// A wave owns 32 co x 16 ci x 9 taps (72 accumulator registers).  With CO 64
// the waves are 2 (co halves) x 2 (ci halves) x 2 (image rows of the step),
// with CO 32 2 (ci) x 4 (row, pixel half); the partial sums of the waves that
// share an output are added up in LDS, so a workgroup makes one atomic per
// weight.  The next step's loads are in flight during a step's MFMAs; one
// barrier a step.  Strides of 88 (x) and 72 (g) pixels put the 16 channels of
// a fragment read in distinct bank groups.
//
// The kernel it replaced took one tap and 32 x 32 channels a workgroup and
// read every operand two bytes at a time: 10.8 ms of the 17.3 ms of a step of
// 8 tiles of 512^2.  This one takes 2.0 ms, some 0.3 PFLOP/s; how that divides
// between the transposing stores to LDS, the loads and the matrix
// instructions has not been measured.
constexpr int WG_T = 512;        // threads
constexpr int WG_XS = 88;        // pixels of a staged x channel: 8 (pixel -1 last), 64, 1, pad
constexpr int WG_GS = 72;        // pixels of a staged g channel: 64, pad
constexpr int WG_XROW = 32 * WG_XS;
__device__ inline uint32_t pair_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ inline uint32_t pair_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// EDGE: W % 64 or H % 2.  Beyond the right edge and below the last row g is
// staged as zeros; x is not zero there for the taps that move the last pixel
// or row in, and may be infinite, so those products are left out (2 to 12 % of
// such a launch).
template <int CO, bool EDGE>
__global__ __launch_bounds__(WG_T) __attribute__((amdgpu_waves_per_eu(4))) void k_conv3x3_wgrad(
    ConvIn ci, const uint16_t* __restrict__ g, float* __restrict__ dw, int N, int H, int W, int Cout,
    int rows) {
    constexpr int GROW = CO * WG_GS, X_N = 6 * WG_XROW, G_N = 4 * GROW;
    constexpr int RED_N = 4 * 18 * 256 * 2;  // partial sums of four waves, in bf16 words
    constexpr int SM_N = X_N + G_N > RED_N ? X_N + G_N : RED_N;
    __shared__ __align__(16) uint16_t smem[SM_N];
    uint16_t* const xt = smem;        // [6 ring slots][32 ci][WG_XS]
    uint16_t* const gt = smem + X_N;  // [2 steps][2 rows][CO][WG_GS]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Cin = ci.C1 + ci.C2;
    const int segs = (W + 63) / 64, blocks_y = (H + rows - 1) / rows;
    const int seg = blockIdx.x % segs, yb = (blockIdx.x / segs) % blocks_y;
    const int n = blockIdx.x / (segs * blocks_y);
    const int x0 = seg * 64, y0 = yb * rows, y1 = min(y0 + rows, H);
    const int co0 = blockIdx.y * CO, ci0 = blockIdx.z * 32;

    // This thread's part of the staging of two rows: 4 pixels x 8 channels of
    // x (threads 0-127), of g (the next 2 CO x 2), or 8 channels of a pixel
    // beside the segment (16 more).
    constexpr int XT = 128, GT = 4 * CO;  // 2 rows x 16 pixel groups x channels / 8
    static_assert(XT + GT + 16 <= WG_T, "a task a thread");
    const bool is_x = tid < XT, is_g = tid >= XT && tid < XT + GT;
    const bool is_h = tid >= XT + GT && tid < XT + GT + 16;
    int trow, tpx, tc;
    if (is_g) {
        const int i = tid - XT;
        tc = i % (CO / 8);
        tpx = 4 * ((i / (CO / 8)) & 15);
        trow = i / (2 * CO);
    } else if (is_h) {
        const int i = tid - XT - GT;
        tc = i & 3;
        tpx = (i >> 2) & 1 ? 64 : -1;
        trow = i >> 3;
    } else {
        tc = tid & 3;
        tpx = 4 * ((tid >> 2) & 15);
        trow = (tid >> 6) & 1;
    }
    // the block's 32 input channels lie in one of the two inputs
    const bool first = ci0 < ci.C1;
    const uint16_t* const xsrc = first ? ci.in1 : ci.in2;
    const int xc = first ? ci.C1 : ci.C2, up = first ? ci.up1 : 0;
    const int xo = (first ? ci0 : ci0 - ci.C1) + 8 * tc;
    const int Hx = up ? (H + 1) / 2 : H, Wx = up ? (W + 1) / 2 : W;
    uint4 v[4];
    // rows y (x: row y0 - 1 + 2 s + trow with s counted two rows ahead of g's)
    auto load = [&](int xrow, int grow) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = make_uint4(0u, 0u, 0u, 0u);
        if (is_g) {
            const int y = grow + trow;
            if (y >= y1) return;
            const uint16_t* p = g + (((size_t)n * H + y) * W + x0 + tpx) * Cout + co0 + 8 * tc;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (x0 + tpx + j < W) v[j] = *reinterpret_cast<const uint4*>(p + (size_t)j * Cout);
        } else if (is_x || is_h) {
            const int y = xrow + trow;
            if (y < 0 || y >= H) return;
            const uint16_t* p = xsrc + ((size_t)n * Hx + (up ? y / 2 : y)) * Wx * xc + xo;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int x = x0 + tpx + j;
                if (x >= 0 && x < W && (is_x || j == 0))
                    v[j] = *reinterpret_cast<const uint4*>(p + (size_t)(up ? x / 2 : x) * xc);
            }
        }
    };
    // slot: ring slot of the first of the two x rows; buf: g's step parity
    auto store = [&](int slot, int buf) {
        if (is_h) {
            const int s = slot + trow;
            uint16_t* d = xt + (s >= 6 ? s - 6 : s) * WG_XROW + 8 * tc * WG_XS + 8 + tpx;
            const uint32_t u[4] = {v[0].x, v[0].y, v[0].z, v[0].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) d[e * WG_XS] = (uint16_t)(u[e >> 1] >> (16 * (e & 1)));
            return;
        }
        if (!is_x && !is_g) return;
        const int s = slot + trow;
        uint16_t* d = is_x ? xt + (s >= 6 ? s - 6 : s) * WG_XROW + 8 * tc * WG_XS + 8 + tpx
                           : gt + (2 * buf + trow) * GROW + 8 * tc * WG_GS + tpx;
        const int stride = is_x ? WG_XS : WG_GS;
        const uint32_t u[4][4] = {{v[0].x, v[0].y, v[0].z, v[0].w}, {v[1].x, v[1].y, v[1].z, v[1].w},
                                  {v[2].x, v[2].y, v[2].z, v[2].w}, {v[3].x, v[3].y, v[3].z, v[3].w}};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            *reinterpret_cast<uint2*>(d + 2 * k * stride) =
                make_uint2(pair_lo(u[0][k], u[1][k]), pair_lo(u[2][k], u[3][k]));
            *reinterpret_cast<uint2*>(d + (2 * k + 1) * stride) =
                make_uint2(pair_hi(u[0][k], u[1][k]), pair_hi(u[2][k], u[3][k]));
        }
    };

    // this wave's share: ci half, then co half and row (CO 64) or row and
    // pixel half (CO 32)
    const int wci = wave & 1, wrow = CO == 64 ? wave >> 2 : (wave >> 1) & 1;
    const int wco = CO == 64 ? (wave >> 1) & 1 : 0;
    const int c_lo = CO == 64 ? 0 : wave >> 2, c_hi = CO == 64 ? 2 : c_lo + 1;
    const int row = lane & 15, kb = lane >> 4;
    f32x4 acc[9][2];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[t][q] = f32x4{0.f, 0.f, 0.f, 0.f};

    // x rows y0 - 1 .. y0 + 2 and g rows y0, y0 + 1 to begin with
    load(y0 - 1, y1);
    store(0, 0);
    load(y0 + 1, y0);
    store(2, 0);
    __syncthreads();
    int slot = 0;  // ring slot of x row y - 1
    for (int y = y0, buf = 0; y < y1; y += 2, buf ^= 1) {
        const bool more = y + 2 < y1;
        if (more) load(y + 3, y + 2);
        const uint16_t* gr = gt + (2 * buf + wrow) * GROW + (32 * wco + row) * WG_GS + 8 * kb;
        for (int c = EDGE && y + wrow >= y1 ? c_hi : c_lo; c < c_hi; ++c) {
            bf16x8 a[2];
#pragma unroll
            for (int q = 0; q < 2; ++q)
                a[q] = as_bf16x8(*reinterpret_cast<const uint4*>(gr + 16 * q * WG_GS + 32 * c));
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                int sl = slot + wrow + dy;
                if (sl >= 6) sl -= 6;
                const uint16_t* xr = xt + sl * WG_XROW + (16 * wci + row) * WG_XS + 8 + 32 * c + 8 * kb;
                const uint4 m = *reinterpret_cast<const uint4*>(xr);
                const uint32_t pv = *reinterpret_cast<const uint32_t*>(xr - 2);
                const uint32_t nx = *reinterpret_cast<const uint32_t*>(xr + 8);
                const uint32_t s0 = __builtin_amdgcn_alignbit(m.x, pv, 16);
                const uint32_t s1 = __builtin_amdgcn_alignbit(m.y, m.x, 16);
                const uint32_t s2 = __builtin_amdgcn_alignbit(m.z, m.y, 16);
                const uint32_t s3 = __builtin_amdgcn_alignbit(m.w, m.z, 16);
                const uint32_t s4 = __builtin_amdgcn_alignbit(nx, m.w, 16);
                uint4 u0 = make_uint4(s0, s1, s2, s3);  // pixel - 1
                if (EDGE && (uint32_t)(W - x0 - 32 * c) < 32u) {
                    int end = W - x0 - 32 * c;
                    asm volatile("" : "+s"(end));  // (masks kept for the three rows would spill)
                    const int e = end - 8 * kb;
                    const uint32_t keep = (e & 1) ? 0xffffu : 0xffff0000u;
                    if (e >> 1 == 0) u0.x &= keep;
                    if (e >> 1 == 1) u0.y &= keep;
                    if (e >> 1 == 2) u0.z &= keep;
                    if (e >> 1 == 3) u0.w &= keep;
                }
                const bf16x8 b0 = as_bf16x8(u0);
                const bf16x8 b1 = as_bf16x8(m);
                const bf16x8 b2 = as_bf16x8(make_uint4(s1, s2, s3, s4));  // pixel + 1
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    acc[3 * dy][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q], b0, acc[3 * dy][q], 0, 0, 0);
                    acc[3 * dy + 1][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q], b1, acc[3 * dy + 1][q], 0, 0, 0);
                    acc[3 * dy + 2][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q], b2, acc[3 * dy + 2][q], 0, 0, 0);
                }
            }
        }
        // rows no wave reads in this step: x ring slots 4 and 5 on, the other
        // g buffer (both last read before the barrier that began the step)
        if (more) store(slot + 4 >= 6 ? slot - 2 : slot + 4, buf ^ 1);
        __syncthreads();
        slot = slot + 2 >= 6 ? slot - 4 : slot + 2;
    }

    // partial sums of the waves with the same output: CO 64 waves 4-7 into
    // 0-3; CO 32 waves 4-7 into 0-3, then 2, 3 into 0, 1
    f32x4* const red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int half = 4; half >= (CO == 64 ? 4 : 2); half >>= 1) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int q = 0; q < 2; ++q) red[((wave - half) * 18 + 2 * t + q) * 64 + lane] = acc[t][q];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int q = 0; q < 2; ++q) acc[t][q] += red[(wave * 18 + 2 * t + q) * 64 + lane];
        }
        __syncthreads();
    }
    if (wave >= (CO == 64 ? 4 : 2)) return;
    // accumulator row 4 kb + r = output channel, column = input channel
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                atomicAdd(&dw[((size_t)t * Cout + co0 + 32 * wco + 16 * q + 4 * kb + r) * Cin + ci0 +
                              16 * wci + row],
                          acc[t][q][r]);
}

// ---- elementwise / small kernels ------------------------------------------

#define GRID_STRIDE(i, n)                                                               \
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (long long)(n); \
         i += (long long)gridDim.x * blockDim.x)

// 2x2 average pooling, NHWC bf16 (H, W even).
__global__ void k_avgpool2(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int N,
                           int H, int W, int C) {
    const int Ho = H / 2, Wo = W / 2;
    GRID_STRIDE(i, (long long)N * Ho * Wo * C) {
        const int c = (int)(i % C);
        long long p = i / C;
        const int x = (int)(p % Wo);
        p /= Wo;
        const int y = (int)(p % Ho);
        const int n = (int)(p / Ho);
        const size_t b = (((size_t)n * H + 2 * y) * W + 2 * x) * C + c;
        const float s = bf2f(in[b]) + bf2f(in[b + C]) + bf2f(in[b + (size_t)W * C]) +
                        bf2f(in[b + (size_t)W * C + C]);
        out[i] = f2bf(0.25f * s);
    }
}

// Gradient of the 2x2 average pool, added to `dx` (fp32, full resolution).
__global__ void k_avgpool2_back(const float* __restrict__ dy, float* __restrict__ dx, int N, int H,
                                int W, int C) {
    GRID_STRIDE(i, (long long)N * H * W * C) {
        const int c = (int)(i % C);
        long long p = i / C;
        const int x = (int)(p % W);
        p /= W;
        const int y = (int)(p % H);
        const int n = (int)(p / H);
        dx[i] += 0.25f * dy[(((size_t)n * (H / 2) + y / 2) * (W / 2) + x / 2) * C + c];
    }
}

// Gradient of nearest 2x upsampling: sum of the 2x2 block (into `dx`, +=).
__global__ void k_upsample2_back(const float* __restrict__ dy, float* __restrict__ dx, int N,
                                 int H, int W, int C, int Ctot, int coff) {
    // dy: [N][H][W][Ctot] (channels coff..coff+C belong to the upsampled input)
    const int Hh = (H + 1) / 2, Wh = (W + 1) / 2;
    GRID_STRIDE(i, (long long)N * Hh * Wh * C) {
        const int c = (int)(i % C);
        long long p = i / C;
        const int x = (int)(p % Wh);
        p /= Wh;
        const int y = (int)(p % Hh);
        const int n = (int)(p / Hh);
        float s = 0.0f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) {
                const int yy = 2 * y + a, xx = 2 * x + b;
                if (yy < H && xx < W) s += dy[(((size_t)n * H + yy) * W + xx) * Ctot + coff + c];
            }
        dx[i] += s;
    }
}

// dx[p][c] (+)= dy[p][coff + c] for c < C (a slice of a concatenated gradient).
__global__ void k_slice_add(const float* __restrict__ dy, float* __restrict__ dx, long long P,
                            int C, int Ctot, int coff, int accumulate) {
    GRID_STRIDE(i, P * C) {
        const long long p = i / C;
        const int c = (int)(i % C);
        const float v = dy[p * Ctot + coff + c];
        dx[i] = accumulate ? dx[i] + v : v;
    }
}

// ReLU backward into bf16 for the next dgrad: g = dy * (act > 0).
__global__ void k_relu_back_bf16(const float* __restrict__ dy, const uint16_t* __restrict__ act,
                                 uint16_t* __restrict__ g, long long n) {
    GRID_STRIDE(i, n) {
        const float v = (act[i] & 0x7fffu) && !(act[i] & 0x8000u) ? dy[i] : 0.0f;
        g[i] = f2bf(v);
    }
}

// ReLU backward and bias gradient in one pass: g = bf16(dy * (act > 0)) and
// db[c] += sum_p g[p][c] (of the rounded g).  C divides the workgroup size
// and the grid stride is a multiple of it, so a thread only ever sees
// channel threadIdx.x % C; a workgroup adds its threads' sums in LDS and
// makes one atomic per channel.
__global__ __launch_bounds__(256) void k_relu_back_bias(const float* __restrict__ dy,
                                                        const uint16_t* __restrict__ act,
                                                        uint16_t* __restrict__ g, long long n,
                                                        int C, float* __restrict__ db) {
    __shared__ float part[256];
    float s = 0.0f;
    GRID_STRIDE(i, n) {
        const float v = (act[i] & 0x7fffu) && !(act[i] & 0x8000u) ? dy[i] : 0.0f;
        const uint16_t b = f2bf(v);
        g[i] = b;
        s += bf2f(b);
    }
    part[threadIdx.x] = s;
    __syncthreads();
    if ((int)threadIdx.x < C) {
        float t = 0.0f;
        for (int k = threadIdx.x; k < (int)blockDim.x; k += C) t += part[k];
        atomicAdd(&db[threadIdx.x], t);
    }
}

// Gradient of an upsampled tensor through its upsampling and the ReLU that
// made it (act): g = bf16(act > 0 ? sum of dy's 2x2 block : 0), dy the first C
// of Ctot channels at twice the size, and the sums of g as dbias partials.
// One pass where k_upsample2_back and k_relu_back_bias took two, and the
// tensor in between was stored: 104 us a call over the three levels of a
// 512^2 x 8 step, where the first of the two alone took 155.  A thread takes 8 channels; 8 * 256 is a multiple of C.
__global__ __launch_bounds__(256) void k_up_relu_back(const float* __restrict__ dy,
                                                      const uint16_t* __restrict__ act,
                                                      uint16_t* __restrict__ g, int N, int H, int W,
                                                      int C, int Ctot, float* __restrict__ dbias) {
    __shared__ float part[4 * 256];
    const int Ho = H / 2, Wo = W / 2, CH = C / 8;
    float sum[8] = {};
    GRID_STRIDE(i, (long long)N * Ho * Wo * CH) {
        const long long p = i / CH;
        const int c = 8 * (int)(i - p * CH);
        const int x = (int)(p % Wo);
        const long long ny = p / Wo;
        const int y = (int)(ny % Ho);
        const size_t n = (size_t)(ny / Ho);
        const float* d = dy + ((n * H + 2 * y) * W + 2 * x) * Ctot + c;
        const size_t off[4] = {0, (size_t)Ctot, (size_t)W * Ctot, (size_t)W * Ctot + Ctot};
        float4 v[4][2];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k][0] = *reinterpret_cast<const float4*>(d + off[k]);
            v[k][1] = *reinterpret_cast<const float4*>(d + off[k] + 4);
        }
        const uint4 a = *reinterpret_cast<const uint4*>(act + p * C + c);
        uint32_t m[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 &q0 = v[0][h], &q1 = v[1][h], &q2 = v[2][h], &q3 = v[3][h];
            m[2 * h] = (uint32_t)f2bf(((q0.x + q1.x) + q2.x) + q3.x) |
                       ((uint32_t)f2bf(((q0.y + q1.y) + q2.y) + q3.y) << 16);
            m[2 * h + 1] = (uint32_t)f2bf(((q0.z + q1.z) + q2.z) + q3.z) |
                           ((uint32_t)f2bf(((q0.w + q1.w) + q2.w) + q3.w) << 16);
        }
        const uint4 r = relu_mask(make_uint4(m[0], m[1], m[2], m[3]), a);
        *reinterpret_cast<uint4*>(g + p * C + c) = r;
        add8(sum, r);
    }
    bias_partials(sum, CH, part, dbias, C, 0);
}

// Gradient of an encoder output through the ReLU that made it: the decoder's
// share (channels coff.. of dcat's Ctot) plus a quarter of the pooled
// tensor's, g = bf16(act > 0 ? dcat + dp / 4 : 0), and dbias partials.  In
// place of k_slice_add, k_avgpool2_back and k_relu_back_bias.
__global__ __launch_bounds__(256) void k_skip_relu_back(const float* __restrict__ dcat, int Ctot,
                                                        int coff, const float* __restrict__ dp,
                                                        const uint16_t* __restrict__ act,
                                                        uint16_t* __restrict__ g, int N, int H,
                                                        int W, int C, float* __restrict__ dbias) {
    __shared__ float part[4 * 256];
    const int CH = C / 8;
    float sum[8] = {};
    GRID_STRIDE(i, (long long)N * H * W * CH) {
        const long long p = i / CH;
        const int c = 8 * (int)(i - p * CH);
        const int x = (int)(p % W);
        const long long ny = p / W;
        const int y = (int)(ny % H);
        const size_t n = (size_t)(ny / H);
        const float4* s = reinterpret_cast<const float4*>(dcat + (size_t)p * Ctot + coff + c);
        const float4* q = reinterpret_cast<const float4*>(
            dp + ((n * (H / 2) + y / 2) * (W / 2) + x / 2) * C + c);
        const float4 s0 = s[0], s1 = s[1], q0 = q[0], q1 = q[1];
        const uint4 a = *reinterpret_cast<const uint4*>(act + p * C + c);
        const uint4 v = make_uint4(
            (uint32_t)f2bf(s0.x + 0.25f * q0.x) | ((uint32_t)f2bf(s0.y + 0.25f * q0.y) << 16),
            (uint32_t)f2bf(s0.z + 0.25f * q0.z) | ((uint32_t)f2bf(s0.w + 0.25f * q0.w) << 16),
            (uint32_t)f2bf(s1.x + 0.25f * q1.x) | ((uint32_t)f2bf(s1.y + 0.25f * q1.y) << 16),
            (uint32_t)f2bf(s1.z + 0.25f * q1.z) | ((uint32_t)f2bf(s1.w + 0.25f * q1.w) << 16));
        const uint4 r = relu_mask(v, a);
        *reinterpret_cast<uint4*>(g + p * C + c) = r;
        add8(sum, r);
    }
    bias_partials(sum, CH, part, dbias, C, 0);
}

// Bias gradients of every layer from their partials.
struct BiasTable {
    static constexpr int MAX = 16;
    const float* part[MAX];
    float* db[MAX];
    int c[MAX];
};
__global__ void k_bias_sum(BiasTable t) {
    const int l = blockIdx.x, c = threadIdx.x;
    if (c >= t.c[l]) return;
    float s = 0.0f;
#pragma unroll 16
    for (int k = 0; k < BIAS_SLOTS; ++k) s += t.part[l][(size_t)k * t.c[l] + c];
    t.db[l][c] += s;
}

// Weights of the data-gradient convolutions of every layer (k_flip_transpose).
struct FlipTable {
    static constexpr int MAX = 16;
    const uint16_t* w[MAX];
    uint16_t* wt[MAX];
    int cout[MAX], cin[MAX];
};
__global__ void k_flip_all(FlipTable t) {
    const int l = blockIdx.y, Cout = t.cout[l], Cin = t.cin[l];
    GRID_STRIDE(i, 9LL * Cout * Cin) {
        // output order: consecutive threads write consecutive words
        const int co = (int)(i % Cout);
        const int r = (int)(i / Cout), ci = r % Cin, tap = r / Cin;
        t.wt[l][i] = t.w[l][((size_t)(8 - tap) * Cout + co) * Cin + ci];
    }
}

// Bias gradient: db[c] += sum_p g[p][c] (g bf16).
__global__ void k_bias_grad(const uint16_t* __restrict__ g, float* __restrict__ db, long long P,
                            int C) {
    // one block per 64-channel group, threads stride over pixels
    const int c = blockIdx.y * 64 + (threadIdx.x & 63);
    const int lanes = blockDim.x / 64;
    float s = 0.0f;
    if (c < C)
        for (long long p = (long long)blockIdx.x * lanes + (threadIdx.x >> 6); p < P;
             p += (long long)gridDim.x * lanes)
            s += bf2f(g[p * C + c]);
    if (c < C) atomicAdd(&db[c], s);
}

// Head: logit[p] = b + sum_c w[c] act[p][c] (1x1 convolution to one
// channel); with `sigmoid` it writes the probability instead.
__global__ void k_head(const uint16_t* __restrict__ act, const float* __restrict__ w,
                       const float* __restrict__ b, float* __restrict__ logit, long long P, int C,
                       int sigmoid) {
    GRID_STRIDE(p, P) {
        float s = b[0];
        // C is a multiple of 32: the pixel's channels as 16-byte loads, summed
        // in channel order
        const uint4* a = reinterpret_cast<const uint4*>(act + p * C);
        for (int c8 = 0; c8 < C / 8; ++c8) {
            const uint4 v = a[c8];
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                s += w[8 * c8 + 2 * k] * bf2f((uint16_t)(u[k] & 0xffffu));
                s += w[8 * c8 + 2 * k + 1] * bf2f((uint16_t)(u[k] >> 16));
            }
        }
        logit[p] = sigmoid ? 1.0f / (1.0f + expf(-s)) : s;
    }
}

// Loss and head gradients: q = sigmoid(logit); binary cross-entropy against
// the target frequency t; dlogit = (q - t) / P.  Writes q, the head weight and
// bias gradients and d(act) in fp32.  loss[0] += sum BCE / P.  C is a
// multiple of 32 up to HEAD_MAX_C: each thread sums its pixels' terms of
// the weight gradient in registers, a workgroup adds them up in LDS and
// makes one atomic per channel.
// MASK: d(act) goes out behind the ReLU that made act, rounded to bf16 (gout),
// with its sums over the pixels in dbias (BIAS_SLOTS partials), instead of
// fp32 into dact.
constexpr int HEAD_MAX_C = 128;
template <int C, bool MASK>
__global__ __launch_bounds__(256) void k_head_back(const uint16_t* __restrict__ act,
                                                   const float* __restrict__ w,
                                                   const float* __restrict__ logit,
                                                   const float* __restrict__ target,
                                                   float* __restrict__ q, float* __restrict__ dact,
                                                   float* __restrict__ dw, float* __restrict__ db,
                                                   float* __restrict__ loss, long long P,
                                                   uint16_t* __restrict__ gout,
                                                   float* __restrict__ dbias) {
    __shared__ float part[C];
    __shared__ float bpart[MASK ? C : 1];
    __shared__ float red[2];
    for (int c = threadIdx.x; c < C; c += blockDim.x) {
        part[c] = 0.0f;
        if (MASK) bpart[c] = 0.0f;
    }
    if (threadIdx.x < 2) red[threadIdx.x] = 0.0f;
    __syncthreads();
    float acc[C], bacc[MASK ? C : 1];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        acc[c] = 0.0f;
        if (MASK) bacc[c] = 0.0f;
    }
    float lsum = 0.0f, bsum = 0.0f;
    GRID_STRIDE(p, P) {
        const float z = logit[p];
        const float qq = 1.0f / (1.0f + expf(-z));
        q[p] = qq;
        const float t = target ? target[p] : 0.0f;
        // BCE with logits, stable form: max(z,0) - z t + log(1 + e^-|z|)
        lsum += fmaxf(z, 0.0f) - z * t + log1pf(expf(-fabsf(z)));
        const float g = (qq - t) / (float)P;
        bsum += g;
        const uint4* a = reinterpret_cast<const uint4*>(act + p * C);
        float4* d = reinterpret_cast<float4*>(dact + p * C);
#pragma unroll
        for (int c8 = 0; c8 < C / 8; ++c8) {
            const uint4 v = a[c8];
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
            uint32_t m[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int c = 8 * c8 + 2 * k;
                acc[c] += g * bf2f((uint16_t)(u[k] & 0xffffu));
                acc[c + 1] += g * bf2f((uint16_t)(u[k] >> 16));
                if (MASK) {
                    m[k] = ((uint32_t)f2bf(g * w[c]) | ((uint32_t)f2bf(g * w[c + 1]) << 16)) &
                           positive_halves(u[k]);
                    bacc[c] += bf2f((uint16_t)(m[k] & 0xffffu));
                    bacc[c + 1] += bf2f((uint16_t)(m[k] >> 16));
                }
            }
            if (MASK) {
                reinterpret_cast<uint4*>(gout + p * C)[c8] = make_uint4(m[0], m[1], m[2], m[3]);
                continue;
            }
            d[2 * c8] = make_float4(g * w[8 * c8], g * w[8 * c8 + 1], g * w[8 * c8 + 2], g * w[8 * c8 + 3]);
            d[2 * c8 + 1] = make_float4(g * w[8 * c8 + 4], g * w[8 * c8 + 5], g * w[8 * c8 + 6],
                                        g * w[8 * c8 + 7]);
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        float v = acc[c];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if ((threadIdx.x & 63) == 0) atomicAdd(&part[c], v);
        if (MASK) {
            float bv = bacc[c];
            for (int off = 32; off > 0; off >>= 1) bv += __shfl_xor(bv, off);
            if ((threadIdx.x & 63) == 0) atomicAdd(&bpart[c], bv);
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        lsum += __shfl_xor(lsum, off);
        bsum += __shfl_xor(bsum, off);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&red[0], lsum);
        atomicAdd(&red[1], bsum);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += blockDim.x) {
        atomicAdd(&dw[c], part[c]);
        if (MASK) atomicAdd(&dbias[(size_t)(blockIdx.x % BIAS_SLOTS) * C + c], bpart[c]);
    }
    if (threadIdx.x == 0) {
        atomicAdd(loss, red[0] / (float)P);
        atomicAdd(db, red[1]);
    }
}

// Adam step on fp32 master weights, refreshing the bf16 copy (may be null).
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, uint16_t* __restrict__ pb, long long n, float lr,
                       float b1, float b2, float eps, float bc1, float bc2) {
    GRID_STRIDE(i, n) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float upd = lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
        const float np = p[i] - upd;
        p[i] = np;
        if (pb) pb[i] = f2bf(np);
    }
}

// fp32 -> bf16 (weights, inputs).
__global__ void k_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, long long n) {
    GRID_STRIDE(i, n) y[i] = f2bf(x[i]);
}

// Weights of the data-gradient convolution: wt[8 - tap][ci][co] = w[tap][co][ci].
__global__ void k_flip_transpose(const uint16_t* __restrict__ w, uint16_t* __restrict__ wt,
                                 int Cout, int Cin) {
    GRID_STRIDE(i, 9LL * Cout * Cin) {
        const int c_in = (int)(i % Cin);
        long long r = i / Cin;
        const int co = (int)(r % Cout);
        const int tap = (int)(r / Cout);
        wt[((size_t)(8 - tap) * Cin + c_in) * Cout + co] = w[i];
    }
}

int grid_for(long long n) {
    long long g = (n + 255) / 256;
    return (int)(g < 1 ? 1 : (g > 65535 ? 65535 : g));
}

}  // namespace

// Tile of k_conv3x3_taps: as many rows as fit into LDS with all channels.
// rows 0: it does not take the channels, or an odd image with an upsampled
// input (whose last pixel's second row or column is outside).
struct TapsTile {
    int rows, block, cw;
};
inline TapsTile conv_taps_tile(int h, int wdt, int c1, int up1, int c2, int cout) {
    auto fits = [&](int rows, int block, int lds) {
        return 2 * conv_taps_words(rows, block, c1, up1, c2) <= lds;
    };
    if (up1 && (h % 2 || wdt % 2)) return {0, 0, 0};
    if (cout % 128 == 0 && fits(4, 128, CT_LDS)) return {4, 128, 2};
    if (cout % 128 == 0 && fits(2, 128, CT_LDS)) return {2, 128, 4};
    if (cout % 64 == 0 && fits(4, 64, CT_LDS)) return {4, 64, 2};
    if (cout % 64 != 0 && cout % 32 == 0 && fits(4, 32, CT_LDS)) return {4, 32, 1};
    return {0, 0, 0};
}
inline bool conv_edge(int h, int wdt) { return wdt % CL_TX != 0 || h % 4 != 0; }
// The LDS-staged convolutions are the faster ones where output channels come
// in blocks of 32, unless most of a large launch would be padding: with at least
// a quarter of its 4 x 64 tiles' pixels in the image (2000 rows of 17 pixels,
// 64 -> 64 channels: 18 us against 32; 8000 rows: 59 against 61), or at most
// two workgroups a CU (8 images of 16 x 16: 12 against 31).  On narrower ones
// the other kernel, whose waves take pixels of several rows, does less.
inline bool lds_conv_applies(int n, int h, int wdt, int c1, int up1, int c2, int cout) {
    // (k_conv3x3_lds numbers the pixels in 32 bits)
    if (cout % 32 != 0 || (long long)n * h * wdt > INT32_MAX) return false;
    if (conv_edge(h, wdt) && c1 + c2 > 32 && conv_taps_tile(h, wdt, c1, up1, c2, cout).rows == 0)
        return false;
    const long long tiles = (long long)n * ((h + 3) / 4) * ((wdt + CL_TX - 1) / CL_TX);
    return 4LL * n * h * wdt >= tiles * 4 * CL_TX ||
           tiles * (cout % 64 == 0 ? cout / 64 : cout / 32) <= 512;
}
// Output channels of one workgroup of the LDS-staged convolution.
inline int lds_conv_block(int cout) { return cout % 64 == 0 ? 64 : 32; }

// Workgroups of 4 x 64 pixels x 64 output channels (two a CU: 210 VGPRs),
// or of 4 x 64 pixels x 32 output channels, three a CU (146 VGPRs, 43.8 KB of
// LDS): a 32-channel layer has few MFMAs per staged byte, so its workgroups
// mostly wait on their loads and stores, and a third one a CU hides more of
// that than taller tiles would save (the three such layers of a 4096^2
// prediction: 891 -> 843 us a call against 8 x 64-pixel tiles at two a CU).
int launch_conv_lds(void* stream, const ConvIn& ci, const uint16_t* w, const float* bias,
                    uint16_t* out, float* outf, const ConvFuse& fz, int n, int h, int wdt, int cout,
                    int relu) {
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool edge = conv_edge(h, wdt), taps = edge && ci.C1 + ci.C2 > 32;
    const TapsTile tile = taps ? conv_taps_tile(h, wdt, ci.C1, ci.up1, ci.C2, cout) : TapsTile{4, 0, 0};
    if (tile.rows == 0) return CAGEO_ERR_ARG;
    const unsigned tiles = (unsigned)n * ((h + tile.rows - 1) / tile.rows) * ((wdt + CL_TX - 1) / CL_TX);
    auto launch = [&](auto kernel, int block, int threads, size_t lds) {
        hipLaunchKernelGGL(kernel, dim3(tiles, cout / block), dim3(threads), lds, st, ci, w, bias, out,
                           outf, fz, n, h, wdt, cout, relu);
    };
    if (taps) {
        auto taps_of = [&](auto kernel, int out_words) {
            const int words = conv_taps_words(tile.rows, tile.block, ci.C1, ci.up1, ci.C2);
            launch(kernel, tile.block, 64 * tile.rows * tile.cw, 2 * (size_t)std::max(words, out_words));
        };
        if (tile.rows == 2) taps_of(k_conv3x3_taps<2, 2, 4>, conv_out_words<2, 2, 4>());
        else if (tile.block == 128) taps_of(k_conv3x3_taps<4, 4, 2>, conv_out_words<4, 4, 2>());
        else if (tile.cw == 2) taps_of(k_conv3x3_taps<2, 4, 2>, conv_out_words<2, 4, 2>());
        else taps_of(k_conv3x3_taps<2, 4, 1>, conv_out_words<2, 4, 1>());
    } else if (cout % 64 == 0) {
        if (edge) launch(k_conv3x3_lds<4, 2, true>, 64, 256, 0);
        else launch(k_conv3x3_lds<4, 2, false>, 64, 256, 0);
    } else {
        if (edge) launch(k_conv3x3_lds<2, 3, true>, 32, 256, 0);
        else launch(k_conv3x3_lds<2, 3, false>, 32, 256, 0);
    }
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

// The backward passes of the trainer: see the kernels.  Channel counts are
// powers of two of at most 256 (the trainer checks); `n` images of h x w.
int nn_dgrad_relu(void* stream, const uint16_t* g, int co, const uint16_t* wt, const uint16_t* act,
                  uint16_t* gout, float* dbias, int n, int h, int w, int cin) {
    const ConvIn ci{g, nullptr, co, 0, 0};
    ConvFuse fz{};
    fz.mask = act;
    fz.dbias = dbias;
    return launch_conv_lds(stream, ci, wt, nullptr, gout, nullptr, fz, n, h, w, cin, 0);
}
int nn_head_back_relu(void* stream, const uint16_t* act, const float* w, const float* logit,
                      const float* target, float* q, uint16_t* gout, float* dw, float* db,
                      float* loss, float* dbias, long long p, int c) {
    if (c != 32) return CAGEO_ERR_ARG;
    const int grid = (int)std::min<long long>(1024, (p + 255) / 256);
    hipLaunchKernelGGL((k_head_back<32, true>), dim3(grid), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), act, w, logit, target, q,
                       (float*)nullptr, dw, db, loss, p, gout, dbias);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}
int nn_up_relu_back(void* stream, const float* dy, const uint16_t* act, uint16_t* g, float* dbias,
                    int n, int h, int w, int c, int ctot) {
    const long long work = (long long)n * (h / 2) * (w / 2) * (c / 8);
    const int grid = (int)std::min<long long>(2048, (work + 255) / 256);
    hipLaunchKernelGGL(k_up_relu_back, dim3(grid), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dy, act, g, n, h, w, c, ctot, dbias);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}
int nn_skip_relu_back(void* stream, const float* dcat, int ctot, int coff, const float* dp,
                      const uint16_t* act, uint16_t* g, float* dbias, int n, int h, int w, int c) {
    const long long work = (long long)n * h * w * (c / 8);
    const int grid = (int)std::min<long long>(2048, (work + 255) / 256);
    hipLaunchKernelGGL(k_skip_relu_back, dim3(grid), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dcat, ctot, coff, dp, act, g, n, h, w,
                       c, dbias);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}
int nn_bias_sums(void* stream, int layers, const float* const* part, float* const* db,
                 const int* c) {
    if (layers > BiasTable::MAX) return CAGEO_ERR_ARG;
    BiasTable t{};
    for (int l = 0; l < layers; ++l) {
        t.part[l] = part[l];
        t.db[l] = db[l];
        t.c[l] = c[l];
    }
    hipLaunchKernelGGL(k_bias_sum, dim3(layers), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), t);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}
int nn_flip_all(void* stream, int layers, const uint16_t* const* w, uint16_t* const* wt,
                const int* cout, const int* cin) {
    if (layers > FlipTable::MAX) return CAGEO_ERR_ARG;
    FlipTable t{};
    for (int l = 0; l < layers; ++l) {
        t.w[l] = w[l];
        t.wt[l] = wt[l];
        t.cout[l] = cout[l];
        t.cin[l] = cin[l];
    }
    hipLaunchKernelGGL(k_flip_all, dim3(128, layers), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), t);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

// The forward convolution with fused consumers wherever the staged kernel
// takes the image (the C ABI's fused call promises whole tiles only): returns
// false, with nothing launched, where it does not.
bool nn_conv3x3_fused(void* stream, const uint16_t* in1, int c1, int up1, const uint16_t* in2,
                      int c2, const uint16_t* w, const float* bias, uint16_t* out, uint16_t* pool,
                      const float* head_w, const float* head_b, float* prob, int head_sigmoid,
                      int n, int h, int wdt, int cout, int relu, int* status) {
    if (!lds_conv_applies(n, h, wdt, c1, up1, c2, cout) || (pool && (h % 2 || wdt % 2)) ||
        (prob && lds_conv_block(cout) != cout))
        return false;
    const ConvIn ci{in1, in2, c1, c2, up1};
    const ConvFuse fz{pool, head_w, head_b, prob, head_sigmoid};
    *status = launch_conv_lds(stream, ci, w, bias, out, nullptr, fz, n, h, wdt, cout, relu);
    return true;
}

}  // namespace cageo

// ---- C ABI ------------------------------------------------------------------
using namespace cageo;

extern "C" {

int cageo_nn_conv3x3(void* stream, const uint16_t* in1, int c1, int up1, const uint16_t* in2,
                     int c2, const uint16_t* w, const float* bias, uint16_t* out, float* outf,
                     int n, int h, int wdt, int cout, int relu) {
    if (!in1 || !w || (!out && !outf) || n <= 0 || h <= 0 || wdt <= 0) return CAGEO_ERR_ARG;
    if (c1 <= 0 || c1 % 32 || c2 < 0 || c2 % 32 || (c2 && !in2) || cout % 16) return CAGEO_ERR_ARG;
    ConvIn ci{in1, in2, c1, c2, up1};
    const long long M = (long long)n * h * wdt;
    if (lds_conv_applies(n, h, wdt, c1, up1, c2, cout))
        return launch_conv_lds(stream, ci, w, bias, out, outf, ConvFuse{}, n, h, wdt, cout, relu);
    // output channel tile: 64 (NT 4), 32 (NT 2) or 16 (NT 1); 4 pixel tiles
    // per wave (256 pixels per workgroup; 8 lowered occupancy and time)
    constexpr int MT = 4;
    const int nt = cout % 64 == 0 ? 4 : (cout % 32 == 0 ? 2 : 1);
    dim3 grid((unsigned)((M + 64 * MT - 1) / (64 * MT)), (unsigned)(cout / (16 * nt)));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (nt == 4)
        hipLaunchKernelGGL((k_conv3x3<4, MT>), grid, dim3(256), 0, s, ci, w, bias, out, outf, n, h,
                           wdt, cout, relu);
    else if (nt == 2)
        hipLaunchKernelGGL((k_conv3x3<2, MT>), grid, dim3(256), 0, s, ci, w, bias, out, outf, n, h,
                           wdt, cout, relu);
    else
        hipLaunchKernelGGL((k_conv3x3<1, MT>), grid, dim3(256), 0, s, ci, w, bias, out, outf, n, h,
                           wdt, cout, relu);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_conv3x3_fusable(int h, int wdt, int cout, int head) {
    if (h <= 0 || wdt <= 0 || cout <= 0 || wdt % CL_TX || h % 4 || cout % 32) return 0;
    return head ? (lds_conv_block(cout) == cout ? 1 : 0) : 1;
}

int cageo_nn_conv3x3_fused(void* stream, const uint16_t* in1, int c1, int up1,
                           const uint16_t* in2, int c2, const uint16_t* w, const float* bias,
                           uint16_t* out, uint16_t* pool, const float* head_w,
                           const float* head_b, float* prob, int head_sigmoid, int n, int h,
                           int wdt, int cout, int relu) {
    if (!in1 || !w || n <= 0 || h <= 0 || wdt <= 0) return CAGEO_ERR_ARG;
    if (c1 <= 0 || c1 % 32 || c2 < 0 || c2 % 32 || (c2 && !in2)) return CAGEO_ERR_ARG;
    if (!out && !pool && !prob) return CAGEO_ERR_ARG;
    if (prob && (out || pool || !head_w || !head_b)) return CAGEO_ERR_ARG;
    if (!cageo_nn_conv3x3_fusable(h, wdt, cout, prob ? 1 : 0)) return CAGEO_ERR_ARG;
    ConvIn ci{in1, in2, c1, c2, up1};
    ConvFuse fz{pool, head_w, head_b, prob, head_sigmoid};
    return launch_conv_lds(stream, ci, w, bias, out, nullptr, fz, n, h, wdt, cout, relu);
}

int cageo_nn_conv3x3_wgrad(void* stream, const uint16_t* in1, int c1, int up1,
                           const uint16_t* in2, int c2, const uint16_t* g, float* dw, int n, int h,
                           int wdt, int cout) {
    if (!in1 || !g || !dw || c1 <= 0 || c1 % 32 || c2 % 32 || cout % 32) return CAGEO_ERR_ARG;
    if (n <= 0 || h <= 0 || wdt <= 0) return CAGEO_OK;  // an empty sum
    ConvIn ci{in1, in2, c1, c2, up1};
    // image rows a workgroup: some 512 workgroups (two a CU), the fewest
    // atomics that fill the chip; at least 4, the ring's extra rows cost 2
    const int co = cout % 64 == 0 ? 64 : 32;
    const long long segs = (wdt + 63) / 64;
    const long long work = segs * n * h * (cout / co) * ((c1 + c2) / 32);
    long long rows = std::min<long long>(std::max<long long>((work + 511) / 512, 4), h);
    rows = (rows + 1) & ~1LL;
    const dim3 grid((unsigned)(segs * n * ((h + rows - 1) / rows)), (unsigned)(cout / co),
                    (unsigned)((c1 + c2) / 32));
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool edge = wdt % 64 != 0 || h % 2 != 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(WG_T), 0, st, ci, g, dw, n, h, wdt, cout, (int)rows);
    };
    if (co == 64 && edge) launch(k_conv3x3_wgrad<64, true>);
    else if (co == 64) launch(k_conv3x3_wgrad<64, false>);
    else if (edge) launch(k_conv3x3_wgrad<32, true>);
    else launch(k_conv3x3_wgrad<32, false>);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_flip_transpose(void* stream, const uint16_t* w, uint16_t* wt, int cout, int cin) {
    hipLaunchKernelGGL(k_flip_transpose, dim3(grid_for(9LL * cout * cin)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), w, wt, cout, cin);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_avgpool2(void* stream, const uint16_t* in, uint16_t* out, int n, int h, int w, int c) {
    if (h % 2 || w % 2) return CAGEO_ERR_ARG;
    hipLaunchKernelGGL(k_avgpool2, dim3(grid_for((long long)n * h * w * c / 4)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), in, out, n, h, w, c);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_avgpool2_back(void* stream, const float* dy, float* dx, int n, int h, int w, int c) {
    hipLaunchKernelGGL(k_avgpool2_back, dim3(grid_for((long long)n * h * w * c)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dy, dx, n, h, w, c);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_upsample2_back(void* stream, const float* dy, float* dx, int n, int h, int w, int c,
                            int ctot, int coff) {
    hipLaunchKernelGGL(k_upsample2_back, dim3(grid_for((long long)n * ((h + 1) / 2) * ((w + 1) / 2) * c)),
                       dim3(256), 0, reinterpret_cast<hipStream_t>(stream), dy, dx, n, h, w, c,
                       ctot, coff);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_slice_add(void* stream, const float* dy, float* dx, long long p, int c, int ctot,
                       int coff, int accumulate) {
    hipLaunchKernelGGL(k_slice_add, dim3(grid_for(p * c)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dy, dx, p, c, ctot, coff, accumulate);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_relu_back(void* stream, const float* dy, const uint16_t* act, uint16_t* g,
                       long long n) {
    hipLaunchKernelGGL(k_relu_back_bf16, dim3(grid_for(n)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dy, act, g, n);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_bias_grad(void* stream, const uint16_t* g, float* db, long long p, int c) {
    dim3 grid((unsigned)std::min<long long>(1024, (p + 3) / 4), (unsigned)((c + 63) / 64));
    hipLaunchKernelGGL(k_bias_grad, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), g,
                       db, p, c);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_head(void* stream, const uint16_t* act, const float* w, const float* b, float* logit,
                  long long p, int c, int sigmoid) {
    if (!act || !w || !b || !logit || p < 0 || c <= 0 || c % 32) return CAGEO_ERR_ARG;
    hipLaunchKernelGGL(k_head, dim3(grid_for(p)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), act, w, b, logit, p, c, sigmoid);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_head_back(void* stream, const uint16_t* act, const float* w, const float* logit,
                       const float* target, float* q, float* dact, float* dw, float* db,
                       float* loss, long long p, int c) {
    if (!act || !w || !logit || !q || !dact || !dw || !db || !loss || p <= 0) return CAGEO_ERR_ARG;
    const int grid = (int)std::min<long long>(1024, (p + 255) / 256);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (c == 32)
        hipLaunchKernelGGL((k_head_back<32, false>), dim3(grid), dim3(256), 0, s, act, w, logit, target, q,
                           dact, dw, db, loss, p, (uint16_t*)nullptr,
                           (float*)nullptr);
    else if (c == 64)
        hipLaunchKernelGGL((k_head_back<64, false>), dim3(grid), dim3(256), 0, s, act, w, logit, target, q,
                           dact, dw, db, loss, p, (uint16_t*)nullptr,
                           (float*)nullptr);
    else if (c == 96)
        hipLaunchKernelGGL((k_head_back<96, false>), dim3(grid), dim3(256), 0, s, act, w, logit, target, q,
                           dact, dw, db, loss, p, (uint16_t*)nullptr,
                           (float*)nullptr);
    else if (c == HEAD_MAX_C)
        hipLaunchKernelGGL((k_head_back<HEAD_MAX_C, false>), dim3(grid), dim3(256), 0, s, act, w, logit,
                           target, q, dact, dw, db, loss, p, (uint16_t*)nullptr,
                           (float*)nullptr);
    else
        return CAGEO_ERR_ARG;
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_relu_back_bias(void* stream, const float* dy, const uint16_t* act, uint16_t* g,
                            long long p, int c, float* db) {
    if (!dy || !act || !g || !db || p <= 0 || c <= 0 || 256 % c) return CAGEO_ERR_ARG;
    const long long n = p * c;
    const long long blocks = std::min<long long>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(k_relu_back_bias, dim3((unsigned)blocks), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), dy, act, g, n, c, db);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_adam(void* stream, float* p, const float* g, float* m, float* v, uint16_t* pb,
                  long long n, float lr, float b1, float b2, float eps, int step) {
    const float bc1 = 1.0f - powf(b1, (float)step), bc2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(grid_for(n)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), p, g, m, v, pb, n, lr, b1, b2, eps,
                       bc1, bc2);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

int cageo_nn_to_bf16(void* stream, const float* x, uint16_t* y, long long n) {
    hipLaunchKernelGGL(k_to_bf16, dim3(grid_for(n)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), x, y, n);
    CAGEO_HIP_TRY(hipGetLastError());
    return CAGEO_OK;
}

}  // extern "C"
