// nn_ops.hip -- neural-network ops of the learned warm start, for gfx950.
//
// Tensors are NHWC; activations bf16, accumulation fp32.  A 3x3 convolution
// (padding 1) is an implicit GEMM: rows m = (n, y, x) pixels, columns output
// channels, K = 9 taps x input channels, on v_mfma_f32_16x16x32_bf16 (A:
// lane i + 16 (k / 8) holds A[i][k], element k % 8; B: lane j + 16 (k / 8)
// holds B[k][j]; C: lane j + 16 (i / 4) holds C[i][j], element i % 4).
// Weights: fp32 masters and gradients [9][Cout][Cin] (tap = 3 ky + kx), bf16
// copies in operand order (conv_weight_index).  The data gradient of a conv is a
// forward conv of the output gradient with the flipped, transposed weights;
// the weight gradient is a split-K GEMM over pixels whose partials are summed
// in a fixed order (deterministic).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nn_ops.h"

#include <algorithm>

namespace cvt {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

__device__ __forceinline__ float bf2f(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ uint16_t f2bf(float f)
{
    return __builtin_bit_cast(uint16_t, (__bf16)f);   // to nearest even, in hardware
}

__device__ __forceinline__ void unpack8(const uint4 &v, float f[8])
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[2 * k] = __uint_as_float(w[k] << 16);
        f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
    }
}
__device__ __forceinline__ uint4 pack8(const float f[8])
{
    bf16x8 v;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (__bf16)f[k];
    const u32x4 w = __builtin_bit_cast(u32x4, v);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// g where the layer's output y > 0, else 0: the derivative of the ReLU
__device__ __forceinline__ uint4 relu_mask(uint4 g, const uint4 &y)
{
    uint32_t w[4] = {g.x, g.y, g.z, g.w};
    const uint32_t yw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!(__uint_as_float(yw[k] << 16) > 0.0f)) w[k] &= 0xffff0000u;
        if (!(__uint_as_float(yw[k] & 0xffff0000u) > 0.0f)) w[k] &= 0x0000ffffu;
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// Implicit-GEMM 3x3 convolution, NHWC bf16, fp32 accumulation on MFMA:
// out[m][co] = act(bias[co] + sum_tap sum_ci in[m + off(tap)][ci] * w[tap][co][ci])
// A wave computes a strip of 16 x R pixels (columns x rows) of 32 output
// channels; the block's WX x WY strips share one input window in LDS.  Every
// sum runs over the taps in order and, within a tap, over 32-channel slices,
// whatever the tile: the rounding of a layer does not depend on the batch.
// The weights are stored in the order of the MFMA's row operand
// (k_weights_bf16) and come straight from memory to registers.  The channels
// of a lane's two row operands interleave by fours, so that a lane ends with
// eight consecutive channels of its pixel: one 16-byte store.
// The input channels come from in0 (the first c0, read at half resolution
// when `up`: the nearest upsampling of a decoder level) and then in1, so a
// skip concatenation needs no tensor of its own.
// The items (tile, 32-channel group) of one tile run on one XCD, next to each
// other: `per` tiles to each of the 8 XCDs.
struct ConvShape {
    int H, W, Cin, Cout, tilesX, tilesY, tiles;
};

// the source of channel slice sl of image n, as a buffer that reads zero
// outside, and byte offset / pitch of its pixels
struct ConvSource {
    __amdgpu_buffer_rsrc_t rsrc;
    int pitch, row, sh;                            // bytes per pixel, pixels per row
};
__device__ __forceinline__ ConvSource conv_source(const NnConv &p, const ConvShape &q, int n, int sl)
{
    const int ci0 = 32 * sl;
    const bool first = ci0 < p.c0;
    const int C = first ? p.c0 : q.Cin - p.c0, sh = first ? p.up : 0;
    const int Hs = q.H >> sh, Ws = q.W >> sh;
    const uint16_t *src = (first ? p.in0 + ci0 : p.in1 + (ci0 - p.c0)) + (long)n * Hs * Ws * C;
    ConvSource c;
    c.rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, 2 * Hs * Ws * C, 0x00020000);
    c.pitch = 2 * C;
    c.row = Ws;
    c.sh = sh;
    return c;
}
// 8 channels from byte o of pixel (yy, xx), zero outside the image
__device__ __forceinline__ u32x4 conv_load(const ConvSource &c, const ConvShape &q, int yy, int xx, int o)
{
    const bool in = (uint32_t)yy < (uint32_t)q.H && (uint32_t)xx < (uint32_t)q.W;
    return __builtin_amdgcn_raw_buffer_load_b128(
        c.rsrc, in ? (uint32_t)(((yy >> c.sh) * c.row + (xx >> c.sh)) * c.pitch + o) : ~0u, 0, 0);
}

// bias, activation and stores of a strip: column x, rows y0 .. of image n,
// channels co .. co + 7 of this lane
template <int R, int NT>
__device__ __forceinline__ void conv_store(const NnConv &p, const ConvShape &q, const f32x4 (&acc)[R][NT],
                                           int n, int y0, int x, int co, int b0 = 0)
{
    static_assert(R % 2 == 0, "rows in pairs");
    float bv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bv[e] = p.bias ? p.bias[co + e] : 0.0f;
    const bool low = co < p.c_low;                 // uniform: c_low is a multiple of 32
    const int Co = q.Cout - p.c_low, Cl = low ? p.c_low : q.Cout;
    const long o0 = ((long)(n * q.H + y0) * q.W + x) * Co + co - p.c_low;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
        uint4 w[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = acc[r + j][b0 + (e >> 2)][e & 3] + bv[e];
                if (p.relu) v[e] = fmaxf(v[e], 0.0f);
            }
            w[j] = pack8(v);
            if (low || x >= q.W || y0 + r + j >= q.H) continue;
            const long o = o0 + (long)(r + j) * q.W * Co;
            uint4 u = w[j];
            if (p.mask && !p.c_low) u = relu_mask(u, *reinterpret_cast<const uint4 *>(p.mask + o));
            *reinterpret_cast<uint4 *>(p.out + o) = u;
        }
        if (!low && !p.pool) continue;
        // 2x2 sums of the rounded values, the right column from the next lane
        float f[2][8], v[8];
        unpack8(w[0], f[0]);
        unpack8(w[1], f[1]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float g[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                g[j] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f[j][e]), 0xb1,
                                                                  0xf, 0xf, true));
            v[e] = f[0][e] + g[0] + f[1][e] + g[1];
            if (!low) v[e] *= 0.25f;
        }
        if (x >= q.W || y0 + r >= q.H || (x & 1)) continue;
        const long o = ((long)(n * (q.H / 2) + (y0 + r) / 2) * (q.W / 2) + x / 2) * Cl + co;
        uint4 u = pack8(v);
        if (low && p.mask) u = relu_mask(u, *reinterpret_cast<const uint4 *>(p.mask + o));
        *reinterpret_cast<uint4 *>((low ? p.low : p.pool) + o) = u;
    }
}

// Convolution of NS slices whose weights stay in registers while the block
// walks over its tiles (one channel group per block).  The pixels of one
// window row at one column offset and slice are one MFMA operand, read once
// and multiplied with the weights of the three vertical taps into three rows
// of sums: 3 (R + 2) LDS reads for 18 R MFMAs per slice.  The next tile's
// window is loaded meanwhile.
// block 64 WX WY, grid 8 J, J a multiple of Cout / 32.
template <int R, int WX, int WY, int NS>
__global__ __launch_bounds__(64 * WX * WY, NS == 1 ? 2 : 1) void k_conv3x3_keep(const NnConv p,
                                                                              const ConvShape q)
{
    constexpr int GT = 64 * WX * WY;
    constexpr int PX = 16 * WX + 2, PY = R * WY + 2;
    constexpr int LK = 40, SL = PX * PY * LK;      // LDS pitch of a pixel, a slice (bf16)
    constexpr int NA = (PX * PY * 4 + GT - 1) / GT;   // 16-byte loads per thread and slice
    __shared__ uint16_t sA[NS * SL];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wx = wave % WX, wy = wave / WX;
    const int NC = q.Cout >> 5, per = (q.tiles + 7) >> 3, J = (gridDim.x >> 3) / NC;
    const int tile0 = (blockIdx.x & 7) * per, mine = min(per, q.tiles - tile0);
    const int cg = (blockIdx.x >> 3) % NC;
    int k = (blockIdx.x >> 3) / NC;
    if (k >= mine) return;

    int wpos[NA];                                  // window row << 8 | column of the loads
#pragma unroll
    for (int r = 0; r < NA; ++r) {
        const int px = (t + GT * r) >> 2;
        wpos[r] = (px / PX) << 8 | px % PX;
    }
    u32x4 va[NS][NA];
    auto load_window = [&](int kk) {
        const int tile = tile0 + kk;
        const int x0 = (tile % q.tilesX) * (16 * WX) - 1;
        const int y0 = ((tile / q.tilesX) % q.tilesY) * (R * WY) - 1, n = tile / (q.tilesX * q.tilesY);
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) {
            const ConvSource c = conv_source(p, q, n, sl);
#pragma unroll
            for (int r = 0; r < NA; ++r)
                va[sl][r] = conv_load(c, q, y0 + (wpos[r] >> 8), x0 + (wpos[r] & 255), 16 * (t & 3));
        }
    };
    load_window(k);
    bf16x8 wr[9][NS][2];
#pragma unroll
    for (int i = 0; i < 18 * NS; ++i)
        wr[i / (2 * NS)][(i >> 1) % NS][i & 1] =
            *reinterpret_cast<const bf16x8 *>(p.w + ((long)cg * (18 * NS) + i) * 512 + 8 * lane);
    const uint16_t *sx = &sA[(wy * R * PX + 16 * wx + (lane & 15)) * LK + 8 * (lane >> 4)];
    for (; k < mine; k += J) {
        __syncthreads();
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int i = t + GT * r;
                if (i < PX * PY * 4)
                    *reinterpret_cast<u32x4 *>(&sA[sl * SL + (i >> 2) * LK + 8 * (i & 3)]) = va[sl][r];
            }
        __syncthreads();
        if (k + J < mine) load_window(k + J);
        f32x4 acc[R][2];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        // window operands (row, column offset, slice) are read D ahead
        constexpr int D = 3, NX = 3 * (R + 2) * NS;
        bf16x8 xr[D + 1];
        auto read = [&](int j) {
            xr[j % (D + 1)] = *reinterpret_cast<const bf16x8 *>(
                sx + j % NS * SL + (j / (3 * NS) * PX + j / NS % 3) * LK);
        };
#pragma unroll
        for (int j = 0; j < D; ++j) read(j);
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            if (j + D < NX) read(j + D);
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                const int o = j / (3 * NS) - dy;
                if (o < 0 || o >= R) continue;
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    acc[o][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        wr[3 * dy + j / NS % 3][j % NS][b], xr[j % (D + 1)], acc[o][b], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const int tile = tile0 + k;
        conv_store<R, 2>(p, q, acc, tile / (q.tilesX * q.tilesY),
                         ((tile / q.tilesX) % q.tilesY) * (R * WY) + wy * R,
                         (tile % q.tilesX) * (16 * WX) + 16 * wx + (lane & 15), 32 * cg + 8 * (lane >> 4));
    }
}

// Convolution of any number of channels to 16 NT of them: the window of all
// slices lies in LDS, loaded at once, and the weights of a step (tap, slice)
// come WD steps ahead of their use: R LDS reads and R NT MFMAs per step.  An
// LDS pixel is 64 bytes, its four 16-byte parts permuted by the column so that
// 16 lanes of adjacent pixels meet distinct banks.
// block 64 WX WY, grid 8 * (tiles / 8) * Cout / (16 NT), LDS (16 WX + 2) (R WY
// + 2) 64 bytes per slice.
template <int R, int WX, int WY, int NT, int WD>
__global__ __launch_bounds__(64 * WX * WY, NT > 2 ? 1 : 2) void k_conv3x3(const NnConv p,
                                                                        const ConvShape q)
{
    static_assert(9 % WD == 0 && WD % 3 == 0, "the rings turn with the steps");
    constexpr int GT = 64 * WX * WY;
    constexpr int PX = 16 * WX + 2, PY = R * WY + 2, SL = PX * PY * 32;
    constexpr int NA = (PX * PY * 4 + GT - 1) / GT;
    extern __shared__ __attribute__((aligned(16))) uint16_t conv_lds[];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wx = wave % WX, wy = wave / WX;
    const int NC = q.Cout / (16 * NT), ns = q.Cin >> 5, per = (q.tiles + 7) >> 3;
    const int k = blockIdx.x >> 3, cg = k % NC;
    const int tile = (blockIdx.x & 7) * per + k / NC;
    if (k / NC >= per || tile >= q.tiles) return;
    const int x0 = (tile % q.tilesX) * (16 * WX), y0 = ((tile / q.tilesX) % q.tilesY) * (R * WY);
    const int n = tile / (q.tilesX * q.tilesY);

    bf16x8 wr[WD][NT];
    const uint16_t *wp = p.w + (long)cg * (NT / 2) * ns * (18 * 512) + 8 * lane;
    auto load_weights = [&](bf16x8 (&f)[NT], int st) {
#pragma unroll
        for (int b = 0; b < NT; ++b)
            f[b] = *reinterpret_cast<const bf16x8 *>(wp + ((b >> 1) * ns * 18 + 2 * st + (b & 1)) * 512);
    };
#pragma unroll
    for (int i = 0; i < WD; ++i) load_weights(wr[i], i);
    // slices whose loads are in flight together, as registers allow
    constexpr int NB = R == 2 || NT > 2 ? 7 : 4;
    for (int sl = 0; sl < ns; sl += NB) {
        u32x4 va[NB][NA];
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            if (sl + h >= ns) break;
            const ConvSource c = conv_source(p, q, n, sl + h);
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int px = (t + GT * r) >> 2, row = px / PX;
                va[h][r] = conv_load(c, q, row < PY ? y0 - 1 + row : -1, x0 - 1 + px % PX, 16 * (t & 3));
            }
        }
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            if (sl + h >= ns) break;
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const int i = t + GT * r, px = i >> 2;
                if (i < PX * PY * 4)
                    *reinterpret_cast<u32x4 *>(
                        &conv_lds[(sl + h) * SL + px * 32 + 8 * ((i & 3) ^ (((px % PX) >> 2) & 3))]) = va[h][r];
            }
        }
    }
    f32x4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    const int col0 = 16 * wx + (lane & 15);
    // step st = tap * ns + sl, operands two steps ahead
    bf16x8 xr[3][R];
    int tap = 0, sl = 0;                           // of the next read
    auto read_step = [&](bf16x8 (&x)[R]) {
        const int col = col0 + tap % 3;
        const uint16_t *a = conv_lds + sl * SL + (wy * R * PX + (tap / 3) * PX + col) * 32 +
                            8 * ((lane >> 4) ^ ((col >> 2) & 3));
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = *reinterpret_cast<const bf16x8 *>(a + r * PX * 32);
        if (++sl == ns) {
            sl = 0;
            tap = min(tap + 1, 8);
        }
    };
    const int steps = 9 * ns;
    read_step(xr[0]);
    read_step(xr[1]);
    for (int st = 0; st < steps; st += 9) {
#pragma unroll
        for (int u = 0; u < 9; ++u) {
            read_step(xr[(u + 2) % 3]);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int b = 0; b < NT; ++b)
                    acc[r][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u % WD][b], xr[u % 3][r],
                                                                        acc[r][b], 0, 0, 0);
            load_weights(wr[u % WD], min(st + u + WD, steps - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int b = 0; b < NT; b += 2)
        conv_store<R, NT>(p, q, acc, n, y0 + wy * R, x0 + col0, 16 * (NT * cg + b) + 8 * (lane >> 4), b);
}

// eight bf16 of one channel at eight consecutive pixels, for 16 channels and
// 32 pixels per wave, from two transposing LDS reads of a [pixel][channel]
// tile: of each 16 lanes, lane i reads four channels of pixel i / 4 and
// receives channel i of the four pixels
__device__ __forceinline__ bf16x8 read_pixels(const uint16_t *lo, const uint16_t *hi)
{
    typedef __attribute__((address_space(3))) bf16x4 lds4;
    const bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)(bf16x4 *)lo);
    const bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4 *)(bf16x4 *)hi);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Weight-gradient partials of a 32 x 32 block of (co, ci), all nine taps:
// part[split][tap][co][ci] = sum over the split's pixels m of
// g[m][co] * in[m + off(tap)][ci], followed in each split by the bias
// partials [co], the sums of g[m][co] (from the blocks of ci = 0 ..).
// The reduction runs over pixels, 32 of one image row per MFMA step.  A block
// walks over 32 x 2R pixel tiles; g and the input window of a tile are staged
// in LDS as they lie in memory, and the transposing LDS reads deliver 8
// consecutive pixels of a channel at any column offset, so every tap reads
// the one window.  Wave w takes 16 output channels (w & 1) of R rows (w / 2):
// a window row's six operands (3 column offsets, 2 x 16 input channels) meet
// the g operands of the three rows it is a vertical neighbour of, 18 MFMAs
// for 14 reads; 72 sums per lane stay in registers over the whole split.  The
// next tile's loads run during a tile's MFMAs.  Pixels outside the image read
// as zero.  LDS rows are 64 bytes per pixel; the two 32-byte halves swap every
// eight columns, which keeps the 32 lanes of a read phase on distinct banks.
// Input channels come as in k_conv3x3.  grid Cout / 32 * Cin / 32 * splits, the
// splits a multiple of 8: the blocks of one split run on one XCD, next to each
// other, so its pixels are read from memory once.
// Bound by memory on large images: 16 images of 256^2, 32 -> 32 channels, 35 us
// for 134 MB (128 us when each tap read its own shifted tile, transposed by
// eight-byte pieces), 96 -> 32 63 us (346 us); the bias gradient was a pass of
// its own over g, 31 us.
template <int R>
__global__ __launch_bounds__(256, 2) void k_conv3x3_dw(const NnConv p, const uint16_t *__restrict__ g,
                                                       float *__restrict__ part, int H, int W,
                                                       int Cin, int Cout, int tilesX, int tilesY,
                                                       int tiles, int splits)
{
    constexpr int TH = 2 * R, PX = 34, PY = TH + 2;
    constexpr int NX = (PX * PY * 4 + 255) / 256, NG = TH * 32 * 4 / 256;
    constexpr int RED = 2 * 64 * 72 * 4;           // bytes of the final sum over row sets
    constexpr int LDS = (PX * PY + TH * 32) * 64;
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS > RED ? LDS : RED];
    uint16_t *sX = reinterpret_cast<uint16_t *>(lds), *sG = sX + PX * PY * 32;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nci = Cin >> 5, P = (Cout >> 5) * nci;
    const int k = blockIdx.x >> 3, pair = k % P;
    const int split = (k / P) * 8 + (blockIdx.x & 7);
    const int co0 = 32 * (pair / nci), ci0 = 32 * (pair % nci);
    const int tb = (int)((long)tiles * split / splits), te = (int)((long)tiles * (split + 1) / splits);
    const int cot = wave & 1, rs = wave >> 1;
    const bool first = ci0 < p.c0;
    const uint16_t *src = first ? p.in0 + ci0 : p.in1 + (ci0 - p.c0);
    const int C = first ? p.c0 : Cin - p.c0, sh = first ? p.up : 0, Hs = H >> sh, Ws = W >> sh;

    // window loads: LDS position | column << 16 | row << 24
    int wpos[NX];
#pragma unroll
    for (int r = 0; r < NX; ++r) {
        const int px = (t + 256 * r) >> 2, col = px % PX, row = px / PX;
        wpos[r] = (px * 32 + 8 * ((t & 3) ^ (2 * ((col >> 3) & 1)))) | col << 16 | row << 24;
    }
    u32x4 vx[NX], vg[NG];
    auto load = [&](int tile) {
        const int x0 = (tile % tilesX) * 32, y0 = ((tile / tilesX) % tilesY) * TH;
        const int n = tile / (tilesX * tilesY);
        const auto rx = __builtin_amdgcn_make_buffer_rsrc((void *)(src + (long)n * Hs * Ws * C), 0,
                                                          2 * Hs * Ws * C, 0x00020000);
        const auto rg = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(g + (long)n * H * W * Cout + co0), 0, 2 * H * W * Cout, 0x00020000);
#pragma unroll
        for (int r = 0; r < NX; ++r) {
            const int yy = y0 - 1 + (wpos[r] >> 24), xx = x0 - 1 + ((wpos[r] >> 16) & 255);
            const uint32_t o = 2 * ((yy >> sh) * Ws + (xx >> sh)) * C + 16 * (t & 3);
            vx[r] = __builtin_amdgcn_raw_buffer_load_b128(
                rx, (uint32_t)yy < (uint32_t)H && (uint32_t)xx < (uint32_t)W ? o : ~0u, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < NG; ++r) {
            const int yy = y0 + 2 * r + (t >> 7), xx = x0 + ((t >> 2) & 31);
            const uint32_t o = 2 * (yy * W + xx) * Cout + 16 * (t & 3);
            vg[r] = __builtin_amdgcn_raw_buffer_load_b128(rg, yy < H && xx < W ? o : ~0u, 0, 0);
        }
    };
    // LDS positions of this lane's reads: column offset dx, pixel half h; the
    // second 16 channels are at ^ 16
    const int pc = 8 * (lane >> 4) + ((lane & 15) >> 2), cc = 4 * (lane & 3);
    int ax[3][2], ag[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int col = pc + 4 * h;
        ag[h] = (rs * R * 32 + col) * 32 + 16 * (cot ^ ((col >> 3) & 1)) + cc;
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
            ax[dx][h] = (rs * R * PX + col + dx) * 32 + 16 * (((col + dx) >> 3) & 1) + cc;
    }
    f32x4 acc[9][2], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[i][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.0f;
    if (tb < te) load(tb);
    for (int tile = tb; tile < te; ++tile) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NX; ++r)
            if (NX * 256 == PX * PY * 4 || t + 256 * r < PX * PY * 4)
                *reinterpret_cast<u32x4 *>(&sX[wpos[r] & 0xffff]) = vx[r];
#pragma unroll
        for (int r = 0; r < NG; ++r)
            *reinterpret_cast<u32x4 *>(
                &sG[((t + 256 * r) >> 2) * 32 + 8 * ((t & 3) ^ (2 * ((t >> 5) & 1)))]) = vg[r];
        __syncthreads();
        if (tile + 1 < te) load(tile + 1);
        // operands are read D steps (of a window row and column offset) ahead
        constexpr int D = 1, NQ = 3 * (R + 2);
        bf16x8 gv[4], xv[D + 1][2];
        auto read_step = [&](int q) {
            const int r = q / 3, dx = q % 3;
#pragma unroll
            for (int b = 0; b < 2; ++b)
                xv[q % (D + 1)][b] = read_pixels(sX + ((ax[dx][0] ^ (16 * b)) + r * PX * 32),
                                                 sX + ((ax[dx][1] ^ (16 * b)) + r * PX * 32));
            if (dx == 0 && r < R) gv[r % 4] = read_pixels(sG + ag[0] + r * 1024, sG + ag[1] + r * 1024);
        };
#pragma unroll
        for (int q = 0; q < D; ++q) read_step(q);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int r = q / 3, dx = q % 3;
            if (q + D < NQ) read_step(q + D);
            if (dx == 0 && r < R)
                accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gv[r % 4], ones, accb, 0, 0, 0);
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                if (r - dy < 0 || r - dy >= R) continue;
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    acc[3 * dy + dx][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        gv[(r - dy) % 4], xv[q % (D + 1)][b], acc[3 * dy + dx][b], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the two row sets' sums
    float *red = reinterpret_cast<float *>(lds);
    __syncthreads();
    if (rs == 1) {
#pragma unroll
        for (int i = 0; i < 72; ++i)
            red[(cot * 72 + i) * 64 + lane] = acc[i >> 3][(i >> 2) & 1][i & 3];
    }
    __syncthreads();
    if (rs == 0) {
        const long sz = (long)Cout * Cin;
        const int co = co0 + 16 * cot + 4 * (lane >> 4), ci = ci0 + (lane & 15);
        float *dst = part + split * (9 * sz + Cout) + (long)co * Cin + ci;
#pragma unroll
        for (int i = 0; i < 72; ++i)
            dst[(i >> 3) * sz + (long)(i & 3) * Cin + 16 * ((i >> 2) & 1)] =
                acc[i >> 3][(i >> 2) & 1][i & 3] + red[(cot * 72 + i) * 64 + lane];
    }
    if (ci0 == 0) {
        __syncthreads();
        if (rs == 1 && (lane & 15) == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) red[16 * cot + 4 * (lane >> 4) + e] = accb[e];
        }
        __syncthreads();
        if (rs == 0 && (lane & 15) == 0) {
            const int c = 16 * cot + 4 * (lane >> 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                part[split * Cout * (9L * Cin + 1) + 9L * Cout * Cin + co0 + c + e] =
                    accb[e] + red[c + e];
        }
    }
}

// out[i] = sum_s part[s][i] in a fixed order (deterministic): a block of 512
// takes 32 consecutive i; its sixteen half waves sum the splits s = q, q + 16,
// ... (q = half wave) in order, then the sums are added in order.
// grid ceil(n / 32).
__global__ __launch_bounds__(512) void k_sum_splits(const float *__restrict__ part, int splits,
                                                    long n, float *__restrict__ out)
{
    __shared__ float red[16][32];
    const int lane = threadIdx.x & 31, q = threadIdx.x >> 5;
    const long i = (long)blockIdx.x * 32 + lane;
    float s = 0.0f;
    if (i < n) {
#pragma unroll 8
        for (int k = q; k < splits; k += 16) s += part[(long)k * n + i];
    }
    red[q][lane] = s;
    __syncthreads();
    if (q == 0 && i < n) {
#pragma unroll
        for (int j = 1; j < 16; ++j) s += red[j][lane];
        out[i] = s;
    }
}

// position of a convolution weight in k_conv3x3's operand order: blocks
// [Cout / 32][9 taps][Cin / 32][2 row operands][64 lanes][8 channels of ci];
// lane l, operand b holds row co = 8 ((l & 15) / 4) + 4 b + l % 4 of its
// 32-channel block and columns ci = 8 (l / 16) ..
__device__ __forceinline__ long conv_weight_index(int tap, int co, int ci, int Cin)
{
    const int c = co & 31, i = ci & 31;
    const int lane = (c >> 3) * 4 + (c & 3) + 16 * (i >> 3), b = (c >> 2) & 1;
    return ((((long)(co >> 5) * 9 + tap) * (Cin >> 5) + (ci >> 5)) * 2 + b) * 512 + lane * 8 + (i & 7);
}

// fp32 master [9][Cout][Cin] -> the bf16 forward copy and the flipped, transposed
// copy for the data gradient (Cin and Cout exchanged, tap -> 8 - tap), both in
// the order of conv_weight_index
__global__ void k_weights_bf16(const float *__restrict__ w, int Cin, int Cout,
                               uint16_t *__restrict__ wf, uint16_t *__restrict__ wb)
{
    const long n = 9L * Cin * Cout;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int tap = (int)(i / ((long)Cin * Cout));
    const int r = (int)(i - (long)tap * Cin * Cout);
    const int co = r / Cin, ci = r - (r / Cin) * Cin;
    const uint16_t v = f2bf(w[i]);
    wf[conv_weight_index(tap, co, ci, Cin)] = v;
    wb[conv_weight_index(8 - tap, ci, co, Cout)] = v;
}

// gradient of the 2x2 average pool, NHWC (H, W even), 8 channels (one 16-byte
// word) per thread with 32-bit indices: channel counts are multiples of 8 and
// every tensor of the network has fewer than 2^31 such words
__global__ void k_avgpool2_bwd(const uint16_t *__restrict__ gout, uint16_t *__restrict__ gin,
                               const uint16_t *__restrict__ mask, int N, int H, int W, int C,
                               int accumulate)
{
    const int C8 = C / 8;
    const int n8 = N * H * W * C8;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const int c8 = i % C8;
    const int p = i / C8;
    const int x = p % W, y = (p / W) % H, b = p / (W * H);
    float v[8], o[8];
    unpack8(reinterpret_cast<const uint4 *>(gout)[((b * (H / 2) + y / 2) * (W / 2) + x / 2) * C8 + c8], v);
    if (accumulate) {
        float g0[8];
        unpack8(reinterpret_cast<const uint4 *>(gin)[i], g0);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = g0[k] + 0.25f * v[k];
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = 0.25f * v[k];
    }
    uint4 w = pack8(o);
    if (mask) w = relu_mask(w, reinterpret_cast<const uint4 *>(mask)[i]);
    reinterpret_cast<uint4 *>(gin)[i] = w;
}

// 1x1 head, one pixel per thread: f[m] = bh + sum_c x[m][c] * wh[.][c], the
// pixel's NN_HEAD_C bf16 channels read as 16-byte words, summed in channel
// order
__global__ void k_head_fwd(const uint16_t *__restrict__ x, const float *__restrict__ wh,
                           const float *__restrict__ bh, float *__restrict__ f, long M)
{
    constexpr int C = NN_HEAD_C;
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    float a = bh[0], b = bh[1];
    const uint4 *src = reinterpret_cast<const uint4 *>(x + m * C);
#pragma unroll
    for (int q = 0; q < C / 8; ++q) {
        const uint4 u = src[q];
        const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = 8 * q + e;
            const float v = bf2f((uint16_t)(wd[e >> 1] >> (16 * (e & 1))));
            a += v * wh[c];
            b += v * wh[C + c];
        }
    }
    f[2 * m] = a;
    f[2 * m + 1] = b;
}

// head gradients: gx[m][c] = sum_j gf[m][j] wh[j][c]; per-split partials of
// dwh[j][c] = sum_m gf[m][j] x[m][c] and dbh[j] = sum_m gf[m][j]; gx is zero
// where x, a ReLU output, is not positive.  A thread takes eight channels (one
// 16-byte load and store, adjacent over the wave) of every 64th pixel of the
// block's split, then each partial is summed by a fixed butterfly over the
// wave and the four waves in order (deterministic).  Bound by memory: 134 MB
// for 16 images of 256^2 in 25 us (42 us with a whole pixel per thread).
__global__ __launch_bounds__(256) void k_head_bwd(const uint16_t *__restrict__ x,
                                                  const float *__restrict__ gf,
                                                  const float *__restrict__ wh,
                                                  uint16_t *__restrict__ gx, float *__restrict__ part,
                                                  long M, long chunk)
{
    constexpr int C = NN_HEAD_C, NP = 2 * C + 2, Q = C / 8;
    __shared__ float red[4][NP];
    const long mb = (long)blockIdx.x * chunk, me = min(M, mb + chunk);
    const int q = threadIdx.x % Q;                 // this thread's 8 channels
    float w0[8], w1[8], acc[18];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        w0[e] = wh[8 * q + e];
        w1[e] = wh[C + 8 * q + e];
    }
#pragma unroll
    for (int k = 0; k < 18; ++k) acc[k] = 0.0f;
    for (long m = mb + threadIdx.x / Q; m < me; m += 256 / Q) {
        const float2 gm = *reinterpret_cast<const float2 *>(gf + 2 * m);
        const uint4 u = *reinterpret_cast<const uint4 *>(x + m * C + 8 * q);
        float v[8], o[8];
        unpack8(u, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o[e] = gm.x * w0[e] + gm.y * w1[e];
            acc[e] += gm.x * v[e];
            acc[8 + e] += gm.y * v[e];
        }
        *reinterpret_cast<uint4 *>(gx + m * C + 8 * q) = relu_mask(pack8(o), u);
        acc[16] += gm.x;
        acc[17] += gm.y;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 18; ++k) {
        float v = acc[k];
#pragma unroll
        for (int o = 32; o >= Q; o >>= 1) v += __shfl_xor(v, o, 64);
        const int c = k < 8 ? 8 * q + k : k < 16 ? C + 8 * q + k - 8 : 2 * C + k - 16;
        if (lane < Q && (k < 16 || q == 0)) red[wave][c] = v;
    }
    __syncthreads();
    if (threadIdx.x < NP) {
        const int k = threadIdx.x;
        part[(long)blockIdx.x * NP + k] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
    }
}

// bilinear sample of the (N, R, R, 2) field at sites u in [0, 1)^2 (pixel
// centres at (i + 0.5) / R, clamped at the border)
__device__ __forceinline__ void bil_coords(float u, int R, int &i0, int &i1, float &t)
{
    float p = u * R - 0.5f;
    p = fminf(fmaxf(p, 0.0f), (float)(R - 1));
    i0 = (int)floorf(p);
    i1 = min(i0 + 1, R - 1);
    t = p - (float)i0;
}

// per site: pred = field(u), loss += |pred - target|^2 * scale, gfield +=
// d loss / d field (atomics; training only)
__global__ void k_sample_loss(const float *__restrict__ field, int R, const float *__restrict__ uv,
                              const float *__restrict__ target, int S, int nb, float scale,
                              float *__restrict__ pred, float *__restrict__ gfield,
                              float *__restrict__ loss_part)
{
    __shared__ float red[256];
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (i < (long)nb * S) {
        const int b = (int)(i / S);
        int x0, x1, y0, y1;
        float tx, ty;
        bil_coords(uv[2 * i], R, x0, x1, tx);
        bil_coords(uv[2 * i + 1], R, y0, y1, ty);
        const float *F = field + (long)b * R * R * 2;
        const float w00 = (1 - tx) * (1 - ty), w10 = tx * (1 - ty), w01 = (1 - tx) * ty, w11 = tx * ty;
        const long p00 = (long)y0 * R + x0, p10 = (long)y0 * R + x1, p01 = (long)y1 * R + x0,
                   p11 = (long)y1 * R + x1;
        float pv[2];
        for (int j = 0; j < 2; ++j)
            pv[j] = w00 * F[2 * p00 + j] + w10 * F[2 * p10 + j] + w01 * F[2 * p01 + j] +
                    w11 * F[2 * p11 + j];
        if (pred) { pred[2 * i] = pv[0]; pred[2 * i + 1] = pv[1]; }
        if (target) {
            const float d0 = pv[0] - target[2 * i], d1 = pv[1] - target[2 * i + 1];
            l = (d0 * d0 + d1 * d1) * scale;
            if (gfield) {
                float *G = gfield + (long)b * R * R * 2;
                const float g0 = 2.0f * d0 * scale, g1 = 2.0f * d1 * scale;
                atomicAdd(&G[2 * p00], w00 * g0); atomicAdd(&G[2 * p00 + 1], w00 * g1);
                atomicAdd(&G[2 * p10], w10 * g0); atomicAdd(&G[2 * p10 + 1], w10 * g1);
                atomicAdd(&G[2 * p01], w01 * g0); atomicAdd(&G[2 * p01 + 1], w01 * g1);
                atomicAdd(&G[2 * p11], w11 * g0); atomicAdd(&G[2 * p11 + 1], w11 * g1);
            }
        }
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0 && loss_part) loss_part[blockIdx.x] = red[0];
}

// Moves each free site of an n x n engine grid by the field sampled at its
// position (displacements in units of the grid side).  A site keeps its
// position when it is fixed, when the target lies off the grid, or when the
// target pixel has zero density (a site there would own no mass).
__global__ void k_apply_disp(float2 *__restrict__ sites, const uint8_t *__restrict__ fixed, int S,
                             const float *__restrict__ field, int R, const float *__restrict__ rho,
                             int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S || fixed[i]) return;
    const float2 s = sites[i];
    const float inv = 1.0f / (float)n;
    int x0, x1, y0, y1;
    float tx, ty;
    bil_coords(s.x * inv, R, x0, x1, tx);
    bil_coords(s.y * inv, R, y0, y1, ty);
    const float w00 = (1 - tx) * (1 - ty), w10 = tx * (1 - ty), w01 = (1 - tx) * ty, w11 = tx * ty;
    const long p00 = (long)y0 * R + x0, p10 = (long)y0 * R + x1, p01 = (long)y1 * R + x0,
               p11 = (long)y1 * R + x1;
    float d[2];
    for (int j = 0; j < 2; ++j)
        d[j] = w00 * field[2 * p00 + j] + w10 * field[2 * p10 + j] + w01 * field[2 * p01 + j] +
               w11 * field[2 * p11 + j];
    const float x = s.x + d[0] * (float)n, y = s.y + d[1] * (float)n;
    if (!(x >= 0.0f && x < (float)n && y >= 0.0f && y < (float)n)) return;   // NaN too
    if (rho[(long)(int)y * n + (int)x] > 0.0f) sites[i] = make_float2(x, y);
}

// Adam (bias-corrected) on fp32 parameters
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m1,
                       float *__restrict__ m2, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.0f - b1) * gi;
    const float v = b2 * m2[i] + (1.0f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = v;
    w[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

__global__ void k_fill_f32(float *__restrict__ p, float v, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// network input at R x R: channel 0 = box-mean density / its mean, channel 1 =
// site count per cell * R^2 / S, channel 2 = 1 where the cell has density;
// channels 3 .. C-1 zero.  The density is n x n with n a multiple of R.
__global__ void k_prepare_density(const float *__restrict__ rho, int n, int R, int C,
                                  const float *__restrict__ inv_mean, uint16_t *__restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)R * R) return;
    const int x = (int)(i % R), y = (int)(i / R);
    const int f = n / R;
    float s = 0.0f;
    for (int yy = 0; yy < f; ++yy)
        for (int xx = 0; xx < f; ++xx) s += rho[(long)(y * f + yy) * n + (x * f + xx)];
    s /= (float)(f * f);
    uint16_t *o = out + i * C;
    o[0] = f2bf(s * inv_mean[0]);
    o[1] = 0;
    o[2] = f2bf(s > 0.0f ? 1.0f : 0.0f);
    for (int c = 3; c < C; ++c) o[c] = 0;
}

// float64 sum of the density: per-block partial sums over a fixed partition,
// then one block adds the partials in index order (deterministic)
__global__ __launch_bounds__(256) void k_rho_partial(const float *__restrict__ rho, long n,
                                                     double *__restrict__ part)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * NN_SUM_BLOCKS)
        acc += (double)rho[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_rho_inv_mean(const double *__restrict__ part, long n,
                                                      float *__restrict__ inv_mean)
{
    __shared__ double red[256];
    red[threadIdx.x] = part[threadIdx.x];
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) inv_mean[0] = red[0] > 0.0 ? (float)((double)n / red[0]) : 0.0f;
}

__global__ void k_prepare_sites(const float *__restrict__ xy, int S, int n, int R, int C,
                                float weight, float *__restrict__ count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S) return;
    const int x = min(max((int)(xy[2 * i] * R / n), 0), R - 1);
    const int y = min(max((int)(xy[2 * i + 1] * R / n), 0), R - 1);
    atomicAdd(&count[(long)y * R + x], weight);
}

// channel 1: the site counts averaged over a (2h+1)^2 window (zero outside
// the grid, divided by the full window area), so the channel holds a local
// site density of about the same noise level at any site count
__global__ void k_prepare_finish(const float *__restrict__ count, int R, int C, int h,
                                 uint16_t *__restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)R * R) return;
    const int x = (int)(i % R), y = (int)(i / R);
    float acc = 0.0f;
    for (int yy = max(y - h, 0); yy <= min(y + h, R - 1); ++yy)
        for (int xx = max(x - h, 0); xx <= min(x + h, R - 1); ++xx) acc += count[(long)yy * R + xx];
    out[i * C + 1] = f2bf(acc / (float)((2 * h + 1) * (2 * h + 1)));
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline unsigned nblk(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// The tile of a convolution.  Bound by memory on large images, by the latency
// of its loads on one; us per call for (channels, side, images):
//   32 -> 32, 256, 16    31 in 32 x 16 tiles            (73 tap by tap)
//              256, 4    12.1, 32 x 8 11.4, 16 x 8 14.4
//              256, 1     7.9,         6.2         6.2
//   64 -> 64, 128, 16    30.6 weights three steps ahead, 34 nine (they take the
//                        registers of a third block), 32 kept   (59)
//   96 -> 96,  64, 16    20.0 nine ahead, 21.4 three, 22.7 kept (33)
//   96 -> 32, 256, 16    73 kept, 93 nine ahead                 (183 and 55
//                        for the concatenated tensor)
//   160 -> 64, 128, 16   67 for 64 channels at once, 84 for 32  (117 + 24)
//               128, 4   18.6                        22.4
//   224 -> 96, 64, 16    31 for 96 channels at once, 47 for 32  (69 + 9)
//               64, 4    26                          17.6
//   96 -> 96,  64, 1      8.4 in 32 x 8 tiles, 6.8 in 16 x 4    (13.5)
//   64 -> 64, 128, 4     10.3                  16
// (in brackets a kernel that staged each tap of 128 pixels by itself).  So the
// largest tile and the most channels at once that still give most of the 256
// CUs a block.  Blocks that keep their weights: two per CU, or one where those
// of three slices take the registers; each then walks its tiles and loads
// ahead (16 images forward, one slice: 0.47 ms, 0.55 with half the blocks).
int nn_conv3x3_kernel(int N, int H, int W, int Cin, int Cout)
{
    const int NC = Cout / 32;
    auto tiles = [&](int tw, int th) { return (long)N * ((W + tw - 1) / tw) * ((H + th - 1) / th); };
    const long t8 = tiles(32, 8);
    if (Cin == 32) return tiles(32, 16) * NC >= 384 ? NN_KEEP_8 : t8 * NC >= 192 ? NN_KEEP_4 : NN_KEEP_2;
    if (Cin == 96 && t8 * NC >= 1024) return NN_KEEP_3SLICES;
    if (Cin >= 128 && Cout % 96 == 0 && t8 * (Cout / 96) >= 192) return NN_CONV_96;
    if (Cin >= 128 && Cout % 64 == 0 && t8 * (Cout / 64) >= 192) return NN_CONV_64;
    if (t8 * NC < 256) return NN_CONV_SMALL;
    return Cin == 64 ? NN_CONV_CIN64 : NN_CONV_32;
}

void nn_conv3x3(hipStream_t s, const NnConv &p, int N, int H, int W, int Cin, int Cout)
{
    const int NC = Cout / 32;
    auto shape = [&](int tw, int th) {
        const int tx = (W + tw - 1) / tw, ty = (H + th - 1) / th;
        return ConvShape{H, W, Cin, Cout, tx, ty, N * tx * ty};
    };
#define NN_KEEP(R, WX, WY, NS)                                                                     \
    {                                                                                              \
        const ConvShape q = shape(16 * WX, R * WY);                                                \
        const int per = (q.tiles + 7) / 8, most = std::max(1, (NS == 1 ? 64 : 32) / NC);           \
        hipLaunchKernelGGL((k_conv3x3_keep<R, WX, WY, NS>), dim3(8 * NC * std::min(per, most)),    \
                           dim3(64 * WX * WY), 0, s, p, q);                                        \
        break;                                                                                     \
    }
#define NN_CONV(R, WX, WY, NT, WD)                                                                 \
    {                                                                                              \
        const ConvShape q = shape(16 * WX, R * WY);                                                \
        const int per = (q.tiles + 7) / 8;                                                         \
        hipLaunchKernelGGL((k_conv3x3<R, WX, WY, NT, WD>), dim3(8 * per * (2 * NC / NT)),          \
                           dim3(64 * WX * WY), (16 * WX + 2) * (R * WY + 2) * 2 * Cin, s, p, q);   \
        break;                                                                                     \
    }
    switch (nn_conv3x3_kernel(N, H, W, Cin, Cout)) {
    case NN_KEEP_8: NN_KEEP(8, 2, 2, 1)
    case NN_KEEP_4: NN_KEEP(4, 2, 2, 1)
    case NN_KEEP_2: NN_KEEP(2, 1, 4, 1)
    case NN_KEEP_3SLICES: NN_KEEP(4, 2, 2, 3)
    case NN_CONV_96: NN_CONV(4, 2, 2, 6, 9)
    case NN_CONV_64: NN_CONV(4, 2, 2, 4, 9)
    case NN_CONV_SMALL: NN_CONV(2, 1, 2, 2, 9)
    case NN_CONV_CIN64: NN_CONV(4, 2, 2, 2, 3)
    default: NN_CONV(4, 2, 2, 2, 9)
    }
#undef NN_CONV
#undef NN_KEEP
}

// rows of a wave in the weight gradient: tiles of 32 x 16 pixels, or 32 x 4
// for so few pixels that the larger ones leave most blocks without one.  A
// training step of 1 / 4 / 16 samples of 256^2 takes 436 / 689 / 1527 us with
// the line at 16384 pixels, 449 / 703 / 1544 at 65536 and 460 / 710 / 1548 at
// 131072.
static int dw_rows(int N, int H, int W)
{
    return (long)N * H * W >= 16384 ? 8 : 2;
}

static int dw_tiles(int N, int H, int W)
{
    const int th = 2 * dw_rows(N, H, W);
    return N * ((H + th - 1) / th) * ((W + 31) / 32);
}

// most pixel splits of a weight gradient: two blocks per CU (in eights: a
// block for each XCD); a 16-sample training step takes 1.71 ms with 512
// blocks, 1.80 with 256 and 1.79 with 768
int nn_dw_max_splits(int Cin, int Cout)
{
    return 8 * std::max(1, 512 / (8 * (Cin / 32) * (Cout / 32)));
}


void nn_conv3x3_dw(hipStream_t s, const NnConv &p, const uint16_t *g, float *dw_db, float *work,
                   int N, int H, int W, int Cin, int Cout)
{
    const int tiles = dw_tiles(N, H, W);
    const int splits = std::min(nn_dw_max_splits(Cin, Cout), 8 * ((tiles + 7) / 8));
    const int P = (Cin / 32) * (Cout / 32), tx = (W + 31) / 32;
    const long n = Cout * (9L * Cin + 1);
    if (dw_rows(N, H, W) == 8)
        hipLaunchKernelGGL((k_conv3x3_dw<8>), dim3(P * splits), dim3(256), 0, s, p, g, work, H, W,
                           Cin, Cout, tx, (H + 15) / 16, tiles, splits);
    else
        hipLaunchKernelGGL((k_conv3x3_dw<2>), dim3(P * splits), dim3(256), 0, s, p, g, work, H, W,
                           Cin, Cout, tx, (H + 3) / 4, tiles, splits);
    hipLaunchKernelGGL(k_sum_splits, dim3(nblk(n, 32)), dim3(512), 0, s, work, splits, n, dw_db);
}

void nn_weights_bf16(hipStream_t s, const float *w, int Cin, int Cout, uint16_t *wf, uint16_t *wb)
{
    hipLaunchKernelGGL(k_weights_bf16, dim3(nblk(9L * Cin * Cout)), dim3(256), 0, s, w, Cin, Cout, wf, wb);
}

void nn_avgpool2_bwd(hipStream_t s, const uint16_t *gout, uint16_t *gin, const uint16_t *mask,
                     int N, int H, int W, int C, int accumulate)
{
    hipLaunchKernelGGL(k_avgpool2_bwd, dim3(nblk((long)N * H * W * C / 8)), dim3(256), 0, s, gout, gin,
                       mask, N, H, W, C, accumulate);
}

void nn_head_fwd(hipStream_t s, const uint16_t *x, const float *wh, const float *bh, float *f,
                 long M)
{
    hipLaunchKernelGGL(k_head_fwd, dim3(nblk(M)), dim3(256), 0, s, x, wh, bh, f, M);
}

int nn_head_splits(long M) { return (int)std::min<long>(1024, std::max<long>(1, M / 1024)); }

void nn_head_bwd(hipStream_t s, const uint16_t *x, const float *gf, const float *wh, uint16_t *gx,
                 float *dwh_db, float *work, long M)
{
    const int splits = nn_head_splits(M);
    const long chunk = (M + splits - 1) / splits;
    constexpr long NP = 2 * NN_HEAD_C + 2;
    hipLaunchKernelGGL(k_head_bwd, dim3(splits), dim3(256), 0, s, x, gf, wh, gx, work, M, chunk);
    hipLaunchKernelGGL(k_sum_splits, dim3(nblk(NP, 32)), dim3(512), 0, s, work, splits, NP, dwh_db);
}

void nn_sample_loss(hipStream_t s, const float *field, int R, const float *uv, const float *target,
                    int S, int nb, float scale, float *pred, float *gfield, float *loss_part)
{
    hipLaunchKernelGGL(k_sample_loss, dim3(nblk((long)nb * S)), dim3(256), 0, s, field, R, uv, target,
                       S, nb, scale, pred, gfield, loss_part);
}

void nn_adam(hipStream_t s, float *w, const float *g, float *m1, float *m2, long n, float lr,
             float b1, float b2, float eps, int t)
{
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_adam, dim3(nblk(n)), dim3(256), 0, s, w, g, m1, m2, n, lr, b1, b2, eps, c1, c2);
}

int nn_splat_halfwidth(int R, int S)
{
    if (S <= 0) return 0;
    return std::max(0, (int)lround((double)R / sqrt((double)S)) - 1);
}

void nn_density_inv_mean(hipStream_t s, const float *rho, int n, double *part, float *inv_mean)
{
    hipLaunchKernelGGL(k_rho_partial, dim3(NN_SUM_BLOCKS), dim3(256), 0, s, rho, (long)n * n, part);
    hipLaunchKernelGGL(k_rho_inv_mean, dim3(1), dim3(256), 0, s, part, (long)n * n, inv_mean);
}

void nn_prepare(hipStream_t s, const float *rho, int n, const float *inv_mean, const float *xy,
                int S, int R, int C, uint16_t *out, float *count)
{
    hipLaunchKernelGGL(k_prepare_density, dim3(nblk((long)R * R)), dim3(256), 0, s, rho, n, R, C,
                       inv_mean, out);
    hipLaunchKernelGGL(k_fill_f32, dim3(nblk((long)R * R)), dim3(256), 0, s, count, 0.0f,
                       (long)R * R);
    if (S > 0)
        hipLaunchKernelGGL(k_prepare_sites, dim3(nblk(S)), dim3(256), 0, s, xy, S, n, R, C,
                           (float)R * R / (float)S, count);
    hipLaunchKernelGGL(k_prepare_finish, dim3(nblk((long)R * R)), dim3(256), 0, s, count, R, C,
                       nn_splat_halfwidth(R, S), out);
}

void nn_apply_disp(hipStream_t s, float2 *sites, const uint8_t *fixed, int S, const float *field,
                   int R, const float *rho, int n)
{
    if (S > 0)
        hipLaunchKernelGGL(k_apply_disp, dim3(nblk(S)), dim3(256), 0, s, sites, fixed, S, field, R,
                           rho, n);
}

}  // namespace cvt
