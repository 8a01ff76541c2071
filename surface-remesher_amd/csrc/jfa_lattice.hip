// jfa_lattice.hip -- the first five JFA passes of a map in one launch.
//
// A pass of step t only moves labels between pixels whose coordinates are
// equal modulo t, and the steps halve: the passes of steps 16 s, 8 s, 4 s,
// 2 s and s never leave a residue class modulo s.  With 16 s the first step
// (the largest power of two below the longer side) a class is a lattice of at
// most 32 x 32 pixels, s apart, so each class runs its five passes alone: one
// wave holds it in registers and no barrier, halo or map is needed between
// the passes.
//
// At 256 pixels per site a class holds about four seeds (Poisson), so a
// wave's state is not a label but a one-hot bit of the class's seeds, ranked
// by label.  The nine taps of a pass are then an OR over a 3 x 3 of words:
// one register OR for the rows and two DPP ORs for the columns (two pixels
// per word), instead of nine table lookups and distances.  Only where some
// OR of the wave holds several seeds are distances compared, one evaluation
// per (pixel, seed of the class) with the seed in scalar registers; in every
// pass but the last, seeds of one column parity only reach the pixels of that
// parity.  Distance and order are the dense pass's (d = fmaf(dy, dy, dx*dx),
// ties to the lower label), so the map equals the five dense passes bit for
// bit.
//
// It replaced a seed scatter and four dense passes, each with its launch, the
// site table staged into every CU's LDS, a map read and a map written.  At 256
// pixels per site the five passes took 23.5 us at 512^2, 52.7 at 2048^2 and
// 350 at 4096^2; the launch takes 12.3, 21.7 and 75 us in an iteration.  It executes 1574 wave
// VALU instructions per class (10.5 us of issue at 2048^2, 42 at 4096^2) and
// is bound by those and, on small grids, by the chain of its latencies (seed
// map load, LDS atomics, site gather, label stores).
//
// Built like jfa.hip with IEEE mode off (no value is ever NaN).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "cvt_finalize.h"
#include "jfa.h"

namespace cvt {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

static constexpr int kLat = 32;      // lattice side of a class
static constexpr int kLatPasses = 5; // passes run on the lattice: steps 16 s .. s
static constexpr int kLatCap = 16;   // seeds of a class on the mask path

// A workgroup of NW waves takes NW neighbouring classes (one row residue, NW
// column residues), so that a lattice point's labels of all its classes are
// one contiguous segment of 4 NW bytes.
template <int NW> struct LatLds {
    // 16 bits per lattice point and class: word 64 r + lane of the class's
    // 512 words, 16 words of skew per four classes so that the four classes a
    // quad of lanes reads lie in different banks
    uint32_t mask[NW * 512 + NW / 4 * 16];
    uint32_t ltab[NW * 32 + NW / 4 * 8];   // label of each ranked seed, then none
    // seeds in order of arrival: label, lattice position, site
    uint32_t lab[NW][kLatCap], pos[NW][kLatCap];
    float2 site[NW][kLatCap];
    int cnt[NW];
    int halt;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t lat_rsrc(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                             0x00020000);
}

// lane + A (row_shl) and lane - A (row_shr) within a row of 16 lanes, 0 from
// outside it
template <int A> __device__ __forceinline__ uint32_t row_shl(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + A, 0xf, 0xf, true);
}
template <int A> __device__ __forceinline__ uint32_t row_shr(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x110 + A, 0xf, 0xf, true);
}

// Lane 16 g + l of a class's wave holds the lattice points of rows 4 r + g
// (r = 0 .. 7) and columns 2 l (low half) and 2 l + 1 (high half) in m[r].
// m becomes the OR of each point's 3 x 3 taps T lattice points apart; taps off
// the lattice are zero (the dense pass redirects them to the centre, which is
// in the set anyway).
template <int T> __device__ __forceinline__ void tap_or(uint32_t (&m)[8], int lane)
{
    uint32_t V[8];
    const int g = lane >> 4;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        if constexpr (T >= 4) {
            constexpr int R = T / 4;
            V[r] = m[r] | (r >= R ? m[r - R] : 0u) | (r + R < 8 ? m[r + R] : 0u);
        } else {
            const uint32_t a = r >= 1 ? m[r - 1] : 0u, b = r + 1 < 8 ? m[r + 1] : 0u;
            if constexpr (T == 2) {
                // rows j +- 2 are the other half's (lane ^ 32): rows r - 1
                // and r of its g + 2 for g < 2, rows r and r + 1 of its g - 2
                // otherwise.  Each half hands over the OR the other wants.
                const uint32_t give = m[r] | (g >= 2 ? a : b);
                V[r] = m[r] | (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (lane ^ 32), (int)give);
            } else {
                // rows j - 1 and j + 1 are the lanes 16 below and above, one
                // register on where they wrap around
                const uint32_t up = g == 3 ? a : m[r], dn = g == 0 ? b : m[r];
                V[r] = m[r] |
                       (uint32_t)__builtin_amdgcn_ds_bpermute(4 * ((lane - 16) & 63), (int)up) |
                       (uint32_t)__builtin_amdgcn_ds_bpermute(4 * ((lane + 16) & 63), (int)dn);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        if constexpr (T >= 2) {
            m[r] = V[r] | row_shl<T / 2>(V[r]) | row_shr<T / 2>(V[r]);
        } else {
            // column 2 l's neighbours are the high halves of lanes l - 1 and
            // l, column 2 l + 1's the low halves of lanes l and l + 1
            const uint32_t side = (row_shr<1>(V[r]) >> 16) | (row_shl<1>(V[r]) << 16);
            m[r] = V[r] | __builtin_amdgcn_alignbit(V[r], V[r], 16) | side;
        }
    }
}

// nonzero where a half of v holds several bits
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t several(uint32_t v)
{
    const u16x2 w = __builtin_bit_cast(u16x2, v) - u16x2{1, 1};
    return v & __builtin_bit_cast(uint32_t, w);
}

__device__ __forceinline__ float lane_f(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// key (d, bit) of a seed for a point whose mask m holds it at bit `at`, above
// every such key where m does not
__device__ __forceinline__ double lat_key(float d, uint32_t m, int at, u32x2 &kv)
{
    const uint32_t in = (uint32_t)__builtin_amdgcn_sbfe((int)m, at, 1);
    kv.y = (in & __float_as_uint(d)) | (~in & 0x7f800000u);
    return __builtin_bit_cast(double, kv);
}

// The halves E of m become the nearest of `seeds` that they hold.  Keys
// (distance, bit) compare as doubles; the bits ascend with the label.
template <int E>
__device__ __forceinline__ void lat_nearest(uint32_t (&m)[8], uint32_t seeds, float vx,
                                                 float vy, float px, const float (&py)[8])
{
    double best[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) best[r] = __hiloint2double(0x7f800000, 0);
#pragma unroll 1
    for (; seeds; seeds &= seeds - 1) {
        const int u = __builtin_ctz(seeds);
        const float dx = lane_f(vx, u) - px, sy = lane_f(vy, u);
        const float a = dx * dx;
        u32x2 kv = {(E ? 0x10000u : 1u) << u, 0u};
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const float dy = sy - py[r];
            best[r] = __builtin_fmin(best[r],
                                     lat_key(__builtin_fmaf(dy, dy, a), m[r], u + 16 * E, kv));
        }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r)
        m[r] = (m[r] & (E ? 0xffffu : 0xffff0000u)) | (uint32_t)__double2loint(best[r]);
}

// A class with more seeds than the mask path takes (sites in step with the
// class stride, or by chance: see jfa_lattice_passes): its five passes by the
// whole workgroup, one dense evaluation per lattice point, between two label
// arrays in the LDS of the masks (which the caller is done with).  1024^2 /
// 6512 sites, where a launch meets such a class most of the time: 50
// iterations 5.10 ms with these passes through the maps, 4.16 in LDS.
template <int NW>
__device__ __forceinline__ void lattice_class_dense(LatLds<NW> &L, const uint32_t *seed,
                                                    const __amdgpu_buffer_rsrc_t rout,
                                                    const float2 *sites, int W, int s, int x0,
                                                    int y0, int nx, int ny)
{
    static_assert(sizeof(L.mask) >= 2 * kLat * kLat * sizeof(uint32_t), "two label arrays");
    const char *sb = reinterpret_cast<const char *>(sites);
    uint32_t *lab[2] = {L.mask, L.mask + kLat * kLat};
    __syncthreads();
    for (int q = threadIdx.x; q < nx * ny; q += blockDim.x)
        lab[0][q] = seed[(size_t)(y0 + s * (q / nx)) * W + (x0 + s * (q % nx))];
    __syncthreads();
#pragma unroll 1
    for (int p = 0; p < kLatPasses; ++p) {
        const uint32_t *in = lab[p & 1];
        uint32_t *dst = lab[~p & 1];
        const int t = 16 >> p;
#pragma unroll 1
        for (int q = threadIdx.x; q < nx * ny; q += blockDim.x) {
            const int j = q / nx, i = q - nx * j;
            const float px = (float)(x0 + s * i) + 0.5f, py = (float)(y0 + s * j) + 0.5f;
            uint32_t l[9];
#pragma unroll
            for (int a = 0; a < 9; ++a) {
                // off-lattice taps are redirected to the point's row or column
                int jj = j + (a / 3 - 1) * t, ii = i + (a % 3 - 1) * t;
                jj = jj < 0 || jj >= ny ? j : jj;
                ii = ii < 0 || ii >= nx ? i : ii;
                l[a] = in[nx * jj + ii];
            }
            double best = __hiloint2double(0x7f800000, -1);
#pragma unroll
            for (int a = 0; a < 9; ++a) {
                const float2 v = *reinterpret_cast<const float2 *>(sb + l[a]);
                const float dx = v.x - px, dy = v.y - py;
                const float d = __builtin_fmaf(dy, dy, dx * dx);
                best = __builtin_fmin(best, __hiloint2double(__float_as_int(d), (int)l[a]));
            }
            const uint32_t lb = (uint32_t)__double2loint(best);
            if (p < kLatPasses - 1)
                dst[q] = lb;
            else
                __builtin_amdgcn_raw_buffer_store_b32(
                    lb, rout, 4u * ((uint32_t)(y0 + s * j) * (uint32_t)W + (uint32_t)(x0 + s * i)),
                    0, 16);
        }
        __syncthreads();
    }
}

// The classes (rx0 .. rx0 + NW - 1, ry) modulo s of one W x H map.
template <int NW>
__device__ __forceinline__ void lattice_group(LatLds<NW> &L, const uint32_t *seed, uint32_t *out,
                                              const float2 *sites, int W, int H,
                                              int s, int rx0, int ry, uint32_t none,
                                              const int *stop)
{
    constexpr int CQ = NW / 4;           // quads of classes
    const int tid = threadIdx.x, lane = tid & 63;
    const int c = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t map_bytes = 4u * (uint32_t)W * (uint32_t)H;
    const __amdgpu_buffer_rsrc_t rin = lat_rsrc(seed, map_bytes), rout = lat_rsrc(out, map_bytes);
    const int ny = (H - ry + s - 1) / s;

    // the group's seeds, each lattice point's classes read four at a time
    // (word by word where a row of odd width ends within them); the stop word
    // of cvt_lloyd_until is loaded beside them, once for the whole workgroup:
    // a finalize beside these passes may be raising it
    if (tid < NW) L.cnt[tid] = 0;
    if (tid == 0) L.halt = stop ? *stop : 0;
    u32x4 v[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int q = it * 64 * NW + tid;
        const int x = rx0 + 4 * (q % CQ) + s * (q / CQ % kLat), j = q / (CQ * kLat);
        const uint32_t off = 4u * ((uint32_t)(ry + s * j) * (uint32_t)W + (uint32_t)x);
        v[it] = u32x4{none, none, none, none};
        if (j < ny && x + 3 < W) {
            v[it] = __builtin_amdgcn_raw_buffer_load_b128(rin, off, 0, 0);
        } else if (j < ny && x < W) {
            v[it].x = __builtin_amdgcn_raw_buffer_load_b32(rin, off, 0, 0);
            if (x + 1 < W) v[it].y = __builtin_amdgcn_raw_buffer_load_b32(rin, off + 4u, 0, 0);
            if (x + 2 < W) v[it].z = __builtin_amdgcn_raw_buffer_load_b32(rin, off + 8u, 0, 0);
        }
    }
    __syncthreads();
    if (L.halt) return;
    // A quad rarely holds two seeds: the lowest label of each of a thread's
    // four quads first, their sites' loads in flight together, then whatever
    // is left one by one.
    const __amdgpu_buffer_rsrc_t rs = lat_rsrc(sites, 0xffffffffu);
    uint32_t lo[4];
    u32x2 st[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        lo[it] = min(min(v[it].x, v[it].y), min(v[it].z, v[it].w));
        st[it] = u32x2{0u, 0u};
        if (lo[it] < none) st[it] = __builtin_amdgcn_raw_buffer_load_b64(rs, lo[it], 0, 0);
    }
    int slot[4], cls[4];
    bool rest = false;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int q = it * 64 * NW + tid;
        cls[it] = 4 * (q % CQ) + (v[it].x == lo[it] ? 0 : v[it].y == lo[it] ? 1 : v[it].z == lo[it] ? 2 : 3);
        slot[it] = kLatCap;
        if (lo[it] < none) {
            slot[it] = atomicAdd(&L.cnt[cls[it]], 1);
            // any other seed of the quad
            const int n = (v[it].x < none) + (v[it].y < none) + (v[it].z < none) + (v[it].w < none);
            rest = rest || n > 1;
        }
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int q = it * 64 * NW + tid;
        if (slot[it] < kLatCap) {
            L.lab[cls[it]][slot[it]] = lo[it];
            L.pos[cls[it]][slot[it]] = (uint32_t)(kLat * (q / (CQ * kLat)) + q / CQ % kLat);
            L.site[cls[it]][slot[it]] = make_float2(__uint_as_float(st[it].x), __uint_as_float(st[it].y));
        }
    }
    if (rest) {
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int q = it * 64 * NW + tid;
            const uint32_t w[4] = {v[it].x, v[it].y, v[it].z, v[it].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (w[e] >= none || w[e] == lo[it]) continue;
                const int cc = 4 * (q % CQ) + e;
                const int k = atomicAdd(&L.cnt[cc], 1);
                if (k >= kLatCap) continue;
                L.lab[cc][k] = w[e];
                L.pos[cc][k] = (uint32_t)(kLat * (q / (CQ * kLat)) + q / CQ % kLat);
                L.site[cc][k] =
                    *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(sites) + w[e]);
            }
        }
    }
    __syncthreads();

    // ---- one class per wave -------------------------------------------------
    const int x0 = rx0 + c;
    const int nx = x0 < W ? (W - x0 + s - 1) / s : 0;
    const int k = __builtin_amdgcn_readfirstlane(L.cnt[c]);
    uint32_t *const mask = L.mask + c * 512 + (c >> 2) * 16;
    uint32_t *const ltab = L.ltab + c * 32 + (c >> 2) * 8;
    if (k <= kLatCap) {
        // seeds ranked by label: lane r holds the seed of rank r
        uint32_t label = lane < k ? L.lab[c][lane] : none;
        int pos = lane < k ? (int)L.pos[c][lane] : 0;
        const float2 st = lane < k ? L.site[c][lane] : make_float2(0.0f, 0.0f);
        int rank = lane < k ? 0 : lane;
        for (int u = 0; u < k; ++u) {
            const uint32_t lu = (uint32_t)__builtin_amdgcn_readlane((int)label, u);
            rank += (lane < k && lu < label) ? 1 : 0;
        }
        label = (uint32_t)__builtin_amdgcn_ds_permute(4 * rank, (int)label);
        pos = __builtin_amdgcn_ds_permute(4 * rank, pos);
        const float vx = __int_as_float(__builtin_amdgcn_ds_permute(4 * rank, __float_as_int(st.x)));
        const float vy = __int_as_float(__builtin_amdgcn_ds_permute(4 * rank, __float_as_int(st.y)));
        if (lane < 32) ltab[lane] = label;
        // the seeds' bits at their lattice points
        const int g = lane >> 4, l = lane & 15;
#pragma unroll
        for (int r = 0; r < 8; ++r) mask[64 * r + lane] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < k) {
            const int i = pos & (kLat - 1), j = pos / kLat;
            reinterpret_cast<uint16_t *>(mask)[2 * (64 * (j >> 2) + 16 * (j & 3) + (i >> 1)) +
                                               (i & 1)] = (uint16_t)(1u << lane);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

        const float px0 = (float)(x0 + s * (2 * l)) + 0.5f;
        const float px1 = (float)(x0 + s * (2 * l + 1)) + 0.5f;
        float py[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) py[r] = (float)(ry + s * (4 * r + g)) + 0.5f;
        const uint32_t all = (1u << k) - 1u;
        const uint32_t odd = (uint32_t)__ballot(lane < k && (pos & 1));
        uint32_t m[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) m[r] = mask[64 * r + lane];
        const bool ragged = nx < kLat || ny < kLat;
        const uint32_t cols = (2 * l < nx ? 0xffffu : 0u) | (2 * l + 1 < nx ? 0xffff0000u : 0u);
#pragma unroll 1
        for (int p = 0; p < kLatPasses; ++p) {
            if (p == 0) tap_or<16>(m, lane);
            else if (p == 1) tap_or<8>(m, lane);
            else if (p == 2) tap_or<4>(m, lane);
            else if (p == 3) tap_or<2>(m, lane);
            else tap_or<1>(m, lane);
            if (ragged) {
#pragma unroll
                for (int r = 0; r < 8; ++r) m[r] &= 4 * r + g < ny ? cols : 0u;
            }
            uint32_t more = 0;
#pragma unroll
            for (int r = 0; r < 8; ++r) more |= several(m[r]);
            // seeds keep their column's parity until the last pass
            const bool last = p == kLatPasses - 1;
            if (__ballot((more & 0xffffu) != 0u))
                lat_nearest<0>(m, last ? all : all & ~odd, vx, vy, px0, py);
            if (__ballot((more & 0xffff0000u) != 0u))
                lat_nearest<1>(m, last ? all : odd, vx, vy, px1, py);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) mask[64 * r + lane] = m[r];
    }
    __syncthreads();

    // ---- the group's labels, four classes of a lattice point per store ------
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int q = it * 64 * NW + tid;
        const int cq = q % CQ, i = q / CQ % kLat, j = q / (CQ * kLat);
        const int x = rx0 + 4 * cq + s * i;
        if (j >= ny || x >= W) continue;
        const int at = 2 * (64 * (j >> 2) + 16 * (j & 3) + (i >> 1)) + (i & 1);
        uint32_t lb[4];
        bool dense = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int cc = 4 * cq + e;
            const uint32_t b =
                reinterpret_cast<const uint16_t *>(L.mask + cc * 512 + cq * 16)[at];
            // the bit's rank, 31 (none) without a bit
            lb[e] = L.ltab[cc * 32 + cq * 8 + __builtin_ctz(b | 0x80000000u)];
            dense = dense || L.cnt[cc] > kLatCap;
        }
        const uint32_t off = 4u * ((uint32_t)(ry + s * j) * (uint32_t)W + (uint32_t)x);
        if (x + 3 < W && !dense) {
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{lb[0], lb[1], lb[2], lb[3]}, rout, off, 0,
                                                   16);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (x + e < W && L.cnt[4 * cq + e] <= kLatCap)
                    __builtin_amdgcn_raw_buffer_store_b32(lb[e], rout, off + 4u * e, 0, 16);
        }
    }
#pragma unroll 1
    for (int cc = 0; cc < NW; ++cc) {
        const int xc = rx0 + cc;
        if (L.cnt[cc] > kLatCap)       // (its pixels lie on the grid: xc < W)
            lattice_class_dense<NW>(L, seed, rout, sites, W, s, xc, ry, (W - xc + s - 1) / s, ny);
    }
}

// blocks go to the 8 XCDs round robin: each XCD takes a contiguous stretch of
// the n groups, so that groups sharing cache lines share an L2
__device__ __forceinline__ int lattice_unit(int b, int n)
{
    const int q8 = n >> 3, r8 = n & 7, xcd = b & 7;
    return xcd * q8 + min(xcd, r8) + (b >> 3);
}

template <int NW>
__global__ __launch_bounds__(64 * NW) void k_jfa_lattice(
    const uint32_t *seed, uint32_t *out, const float2 *__restrict__ sites, int W, int H,
    int s, uint32_t none, const int *__restrict__ stop, int fin,
    const double *__restrict__ blockpart, int *__restrict__ dstate, FinalArgs fa)
{
    __shared__ LatLds<NW> L;
    if (fin && blockIdx.x == 0) {
        // the previous iteration's deferred finalize, beside the passes
        __shared__ double red_e[256], red_g[256];
        cvt_finalize_pending(blockpart, dstate, fa, red_e, red_g);
        return;
    }
    const int u = lattice_unit((int)blockIdx.x - fin, (int)gridDim.x - fin);
    const int gx = s / NW;
    const int ry = u / gx, rx0 = NW * (u - gx * ry);
    if (rx0 >= W) return;
    lattice_group<NW>(L, seed, out, sites, W, H, s, rx0, ry, none, stop);
}

static constexpr int kBatchNW = 8;   // classes per workgroup of the batched launch

__global__ __launch_bounds__(64 * kBatchNW) void k_jfa_batch_lattice(
    const BatchPatch *__restrict__ patches, const int *__restrict__ group_patch,
    const uint32_t *seed, uint32_t *first, const float2 *__restrict__ sites)
{
    __shared__ LatLds<kBatchNW> L;
    const BatchPatch P = patches[group_patch[blockIdx.x]];
    const int s = P.first_step / 16, gx = s / kBatchNW;
    const int u = lattice_unit((int)blockIdx.x - P.lat_off, gx * s);
    const int ry = u / gx, rx0 = kBatchNW * (u - gx * ry);
    if (rx0 >= P.W) return;
    lattice_group<kBatchNW>(L, seed + P.pix_off, first + P.pix_off, sites, P.W, P.H, s, rx0, ry,
                            8u * (uint32_t)(P.site_off + P.cap), nullptr);
}

static int first_step(int W, int H)
{
    int first = 1;
    while (2 * first < std::max(W, H)) first *= 2;
    return first;
}

int jfa_lattice_passes(int W, int H, int S)
{
    const int first = first_step(W, H);
    // steps of 64 and more (a group of four classes is a quad of pixels), a
    // shorter side of at least half the first step (a class is 32 points long
    // and a wave's work does not shrink with its width), and few enough seeds
    // per class: with 8 on average one class in 300 holds more than the mask
    // path's 16, and one or more of them add about 6 us to the launch.  Measured
    // against the dense passes, 50 iterations: 512^2 / 2016 sites (7.9 per
    // class) 2.50 -> 2.42 ms, / 1638 (6.4) 2.46 -> 2.03, 2048^2 / 32263 (7.9)
    // 11.1 -> 9.4, / 26052 (6.4) 10.1 -> 8.2, 1100^2 / 26888 (6.6) 10.4 -> 7.9.
    if (first < 64 || 2 * std::min(W, H) < first) return 0;
    const long classes = (long)(first / 16) * (first / 16);
    return S <= 8 * classes ? kLatPasses : 0;
}

void launch_jfa_lattice(hipStream_t st, const uint32_t *seed, uint32_t *out,
                        const float2 *sites, int W, int H, uint32_t none, const int *stop,
                        const double *blockpart, int *dstate, const FinalArgs *fa)
{
    const int s = first_step(W, H) / 16, fin = fa ? 1 : 0;
    const FinalArgs f = fa ? *fa : FinalArgs();
#define CVT_LATTICE(NW)                                                                        \
    hipLaunchKernelGGL(k_jfa_lattice<NW>, dim3(s / NW * s + fin), dim3(64 * NW), 0, st, seed, \
                       out, sites, W, H, s, none, stop, fin, blockpart, dstate, f)
    // s^2 classes, one per wave.  Wide groups write whole cache lines, narrow
    // ones spread the waves over the CUs and wait for fewer others.  Measured
    // back to back with 4 / 8 / 16 waves: 512^2 11.8 / 14.2 / 20.0 us, 1024^2
    // 14.3 / 15.3 / 18.5, 2048^2 22.9 / 22.2 / 20.6, 4096^2 88 / 65 / 71.
    if (s >= 128)
        CVT_LATTICE(8);
    else if (s >= 64)
        CVT_LATTICE(16);
    else
        CVT_LATTICE(4);
#undef CVT_LATTICE
}

// (a first step of 128 or more: a workgroup's eight classes lie in one stride)
int jfa_batch_lattice_passes(int W, int H, int S)
{
    return first_step(W, H) >= 16 * kBatchNW ? jfa_lattice_passes(W, H, S) : 0;
}

int jfa_batch_lattice_groups(int W, int H)
{
    const int s = first_step(W, H) / 16;
    return s / kBatchNW * s;
}

void launch_jfa_batch_lattice(hipStream_t st, const BatchPatch *patches, const int *group_patch,
                              int groups, const uint32_t *seed, uint32_t *first, const float2 *sites)
{
    if (groups > 0)
        hipLaunchKernelGGL(k_jfa_batch_lattice, dim3(groups), dim3(64 * kBatchNW), 0, st, patches,
                           group_patch, seed, first, sites);
}

}  // namespace cvt
