// raster.hip -- density rasterizer (replaces the reference's discretization_d,
// source/discretization.cu:57-120).
//
// Rule (the reference's, source/discretization.cu:57-85): pixel (tx, ty)
// samples the point (tx * scale, ty * scale) of the shifted UV frame; the first
// triangle in index order whose three float64 barycentric weights are all >= 0
// interpolates the vertex weights, rounded once to float; no hit gives 0.
// Degenerate triangles (zero denominator) never hit.
//
// Instead of testing every triangle at every pixel (O(n^2 F)), triangles are
// binned into 16 x 16 pixel tiles by a conservative bounding box (a counting
// sort: count, prefix sum, fill; linear in the number of (triangle, tile)
// pairs).  A pixel tests its tile's triangles and keeps the lowest-index hit,
// which is the first hit in index order: every triangle holding the sample
// point lists it in that tile.  A triangle so thin that rounding could
// accept points well outside its box (sin^2 of its angle at vertex 1 below
// 1e-12) goes to an "always" list that every pixel tests.  The barycentric
// arithmetic is the oracle's, operation for operation (contraction is off
// for this file).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/cvt.h"
#include "cvt_engine.h"
#include "mesh_scratch.h"

namespace cvt {

#define RT 16   // tile side in pixels

struct TriBox {
    int x0, x1, y0, y1;   // inclusive pixel-index range the triangle may touch; x0 > x1 = none
};

// (triangle, tile) pairs of a pixel box, as tile ranges
__device__ __forceinline__ void tile_range(const TriBox &b, int &tx0, int &tx1, int &ty0, int &ty1)
{
    tx0 = b.x0 / RT; tx1 = b.x1 / RT;
    ty0 = b.y0 / RT; ty1 = b.y1 / RT;
}

// words of a call's status; from ST_PAIRS the (triangle, tile) pairs in 64 bits
enum { ST_BAD, ST_OVERFLOW, ST_ALWAYS, ST_PAIRS = 4, ST_WORDS = 8 };
__device__ __forceinline__ unsigned long long *pair_total(int *status)
{
    return reinterpret_cast<unsigned long long *>(status + ST_PAIRS);
}

// triangle i: index validation and the conservative pixel box.  Triangles to
// test everywhere are appended to alw in any order (a pixel keeps the
// lowest-index hit).
__device__ __forceinline__ TriBox tri_box(const double *__restrict__ pts, int nv,
                                          const int *__restrict__ tri, int i, double scale, int n,
                                          int *__restrict__ alw, int *__restrict__ status)
{
    const int a = tri[3 * i], b = tri[3 * i + 1], c = tri[3 * i + 2];
    TriBox bx = {1, 0, 1, 0};
    if ((unsigned)a >= (unsigned)nv || (unsigned)b >= (unsigned)nv || (unsigned)c >= (unsigned)nv) {
        status[ST_BAD] = 1;
        return bx;
    }
    const double x1 = pts[2 * a], y1 = pts[2 * a + 1];
    const double x2 = pts[2 * b], y2 = pts[2 * b + 1];
    const double x3 = pts[2 * c], y3 = pts[2 * c + 1];
    const double v0x = x2 - x1, v0y = y2 - y1, v1x = x3 - x1, v1y = y3 - y1;
    const double d00 = v0x * v0x + v0y * v0y, d11 = v1x * v1x + v1y * v1y;
    const double d01 = v0x * v1x + v0y * v1y;
    const double den = d00 * d11 - d01 * d01;
    if (den == 0) return bx;                         // never hits
    if (!(den > 1e-12 * d00 * d11)) {                // thin or non-finite: test everywhere
        alw[atomicAdd(&status[ST_ALWAYS], 1)] = i;
        return bx;
    }
    const double xmin = fmin(x1, fmin(x2, x3)), xmax = fmax(x1, fmax(x2, x3));
    const double ymin = fmin(y1, fmin(y2, y3)), ymax = fmax(y1, fmax(y2, y3));
    const double eps = 1e-9 * fmax(xmax - xmin, ymax - ymin) + 1e-300;
    const double lo_x = (xmin - eps) / scale, hi_x = (xmax + eps) / scale;
    const double lo_y = (ymin - eps) / scale, hi_y = (ymax + eps) / scale;
    bx.x0 = (int)fmax(0.0, floor(lo_x));
    bx.x1 = (int)fmin((double)(n - 1), ceil(hi_x));
    bx.y0 = (int)fmax(0.0, floor(lo_y));
    bx.y1 = (int)fmin((double)(n - 1), ceil(hi_y));
    if (!(hi_x >= 0.0) || !(hi_y >= 0.0) || !(lo_x <= n - 1.0) || !(lo_y <= n - 1.0))
        bx = TriBox{1, 0, 1, 0};
    return bx;
}

// per triangle: its box, and its (triangle, tile) pairs counted per tile and
// in all
__global__ void k_tri_boxes(const double *__restrict__ pts, int nv, const int *__restrict__ tri,
                            int nt, double scale, int n, int tiles_x, TriBox *__restrict__ box,
                            int *__restrict__ alw, int *__restrict__ count, int *__restrict__ status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int pairs = 0;
    if (i < nt) {
        const TriBox bx = tri_box(pts, nv, tri, i, scale, n, alw, status);
        box[i] = bx;
        if (bx.x0 <= bx.x1 && bx.y0 <= bx.y1) {
            int tx0, tx1, ty0, ty1;
            tile_range(bx, tx0, tx1, ty0, ty1);
            for (int y = ty0; y <= ty1; ++y)
                for (int x = tx0; x <= tx1; ++x) atomicAdd(&count[y * tiles_x + x], 1);
            pairs = (tx1 - tx0 + 1) * (ty1 - ty0 + 1);
        }
    }
    add_pairs(pairs, pair_total(status));
}

// (triangle, tile) pairs: each triangle writes its index into its tiles'
// lists; with more pairs than the `cap` the list holds, nothing is written and
// the overflow word is raised.
__global__ void k_tile_fill(const TriBox *__restrict__ box, int nt, int tiles_x,
                            const int *__restrict__ start, int *__restrict__ cursor,
                            int *__restrict__ list, int cap, int *__restrict__ status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    if (*pair_total(status) > (unsigned long long)cap) {
        if (i == 0) status[ST_OVERFLOW] = 1;
        return;
    }
    const TriBox b = box[i];
    if (b.x0 > b.x1 || b.y0 > b.y1) return;
    int tx0, tx1, ty0, ty1;
    tile_range(b, tx0, tx1, ty0, ty1);
    for (int y = ty0; y <= ty1; ++y)
        for (int x = tx0; x <= tx1; ++x) {
            const int tile = y * tiles_x + x;
            list[start[tile] + atomicAdd(&cursor[tile], 1)] = i;
        }
}

// LDS written by some lanes of a wave is read by others
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// one wave per tile, four pixels of a column per lane: the lowest-index
// triangle of the tile list and of the "always" list holding the sample point.
// What a triangle's weights take of its corners alone is computed once per
// tile, for kRound triangles at a time, and kept in LDS; a pixel adds its own
// two dot products, tests the signs of the numerators, and divides once, for
// its hit.  host, if set, receives the status and the number of pairs.
// Bound by double-precision arithmetic: 2048^2 pixels, 11858 triangles (five
// candidates per tile) 44 us; 47 us with divisions for every candidate not
// ruled out, 52 us with a pixel per thread, 66 us when every pixel computed
// every triangle in full.
constexpr int kRound = 16;
__global__ __launch_bounds__(256) void k_raster(const double *__restrict__ pts,
                                                const double *__restrict__ wt,
                                                const int *__restrict__ tri,
                                                const int *__restrict__ list,
                                                const int *__restrict__ start,
                                                const int *__restrict__ alw, int tiles_x,
                                                int ntiles, double scale, int n,
                                                float *__restrict__ density,
                                                int *__restrict__ status, int *__restrict__ host)
{
    struct Cand {
        double x1, y1, v0x, v0y, v1x, v1y, d00, d01, d11, den;
    };
    __shared__ Cand cands[4][kRound];
    __shared__ int ids[4][kRound];
    if (host && blockIdx.x == 0 && threadIdx.x == 0) {
        host[0] = status[ST_BAD];
        host[1] = status[ST_OVERFLOW];
        host[2] = pairs_word(*pair_total(status));
    }
    if (status[ST_BAD] || status[ST_OVERFLOW]) return;
    const int wave = threadIdx.x >> 6, t = threadIdx.x & 63;
    const int tile = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + wave);
    if (tile >= ntiles) return;
    Cand *cand = cands[wave];
    int *id = ids[wave];
    const int tx = (tile % tiles_x) * RT + (t & (RT - 1));
    const int ty = (tile / tiles_x) * RT + (t / RT);   // and every fourth row
    const int a = start[tile], len = start[tile + 1] - a, all = len + status[ST_ALWAYS];
    const double x = tx * scale;
    double y[4], h2[4], h3[4], hd[4];
    int hit[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        y[r] = (ty + 4 * r) * scale;
        h2[r] = h3[r] = 0.0;
        hd[r] = 1.0;
        hit[r] = -1;
    }
    for (int j0 = 0; j0 < all; j0 += kRound) {
        const int m = min(kRound, all - j0);
        wave_lds_sync();
        if (t < m) {
            const int j = j0 + t, i = (j < len) ? list[a + j] : alw[j - len];
            const int p1 = tri[3 * i], p2 = tri[3 * i + 1], p3 = tri[3 * i + 2];
            Cand c;
            c.x1 = pts[2 * p1];
            c.y1 = pts[2 * p1 + 1];
            c.v0x = pts[2 * p2] - c.x1;
            c.v0y = pts[2 * p2 + 1] - c.y1;
            c.v1x = pts[2 * p3] - c.x1;
            c.v1y = pts[2 * p3 + 1] - c.y1;
            c.d00 = c.v0x * c.v0x + c.v0y * c.v0y;
            c.d01 = c.v0x * c.v1x + c.v0y * c.v1y;
            c.d11 = c.v1x * c.v1x + c.v1y * c.v1y;
            c.den = c.d00 * c.d11 - c.d01 * c.d01;
            cand[t] = c;
            id[t] = i;
        }
        wave_lds_sync();
        for (int j = 0; j < m; ++j) {
            const Cand c = cand[j];
            const int i = id[j];
            if (c.den == 0) continue;
            const double v2x = x - c.x1, ax = v2x * c.v0x, bx = v2x * c.v1x;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (hit[r] >= 0 && i > hit[r]) continue;   // a lower-index hit is known
                const double v2y = y[r] - c.y1;
                const double d20 = ax + v2y * c.v0y;
                const double d21 = bx + v2y * c.v1y;
                const double n2 = c.d11 * d20 - c.d01 * d21;
                const double n3 = c.d00 * d21 - c.d01 * d20;
                const int in = inside_sign(n2, n3, c.den);
                if (in == 0 || (in < 0 && !inside_exact(n2, n3, c.den))) continue;
                hit[r] = i;
                h2[r] = n2; h3[r] = n3; hd[r] = c.den;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (tx >= n || ty + 4 * r >= n) continue;
        float res = 0.0f;
        if (hit[r] >= 0) {
            const int *p = tri + 3 * hit[r];
            const double b2 = h2[r] / hd[r], b3 = h3[r] / hd[r], b1 = 1.0 - b2 - b3;
            res = (float)(b1 * wt[p[0]] + b2 * wt[p[1]] + b3 * wt[p[2]]);
        }
        density[(long)(ty + 4 * r) * n + tx] = res;
    }
}

}  // namespace cvt

using namespace cvt;

#define RCHK(call, what)                                                                  \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess) return fail(CVT_ERR_HIP, "%s: %s", what, hipGetErrorString(e_)); \
    } while (0)

// One pass over the triangles and one over the pixels, with one wait at the
// end: the lists get room for eight pairs per triangle and one per tile, and a
// mesh with more is seen at the wait, and its lists are filled again with room
// for all.  Arguments in memory of the device are used where they are.
extern "C" int cvt_rasterize(const double *points, const double *weight, int num_point,
                             const int *triangle, int num_tri, float *density, double scale, int n)
{
    clear_error();
    if (n < 1 || n > 16384) return fail(CVT_ERR_ARG, "n = %d outside [1, 16384]", n);
    if (num_point < 0 || num_tri < 0) return fail(CVT_ERR_ARG, "negative sizes");
    if (!density || (num_point > 0 && (!points || !weight)) || (num_tri > 0 && !triangle))
        return fail(CVT_ERR_ARG, "null array");
    if (!(scale > 0.0) || !isfinite(scale)) return fail(CVT_ERR_ARG, "scale %g", scale);
    const int tiles_x = (n + RT - 1) / RT, ntiles = tiles_x * tiles_x;
    hipStream_t st = nullptr;   // the legacy default stream, as the reference's calls use
    const size_t nva = (size_t)std::max(num_point, 1), nta = (size_t)std::max(num_tri, 1);
    const size_t npx = (size_t)n * n;
    const bool own_pts = num_point > 0 && in_place(points, 8);
    const bool own_wt = num_point > 0 && in_place(weight, 8);
    const bool own_tri = num_tri > 0 && in_place(triangle, 4);
    const bool own_den = in_place(density, 4) && !overlap(density, 4 * npx, points, 16 * nva) &&
                         !overlap(density, 4 * npx, weight, 8 * nva) &&
                         !overlap(density, 4 * npx, triangle, 12 * nta);
    double *d_pts = nullptr, *d_wt = nullptr;
    int *d_tri = nullptr, *d_list = nullptr, *d_count = nullptr, *d_start = nullptr,
        *d_cursor = nullptr, *d_alw = nullptr, *d_status = nullptr;
    TriBox *d_box = nullptr;
    float *d_den = nullptr;
    size_t cap = std::min<size_t>(8 * nta + ntiles, INT32_MAX);
    MeshScratch mem;
    Carver carve;
    size_t zeroed = 0;
    auto layout = [&]() {
        carve.base = mem.base();
        carve.at = 0;
        carve(d_status, ST_WORDS);               // zeroed from here
        carve(d_count, ntiles); carve(d_cursor, ntiles);
        zeroed = (carve.at + 255) & ~(size_t)255;
        carve(d_start, (size_t)ntiles + 1); carve(d_box, nta); carve(d_alw, nta);
        if (!own_pts) carve(d_pts, 2 * nva);
        if (!own_wt) carve(d_wt, nva);
        if (!own_tri) carve(d_tri, 3 * nta);
        if (!own_den) carve(d_den, npx);
        carve(d_list, cap);
    };
    layout();
    RCHK(mem.take(carve.at), "alloc");
    layout();
    if (own_pts) d_pts = const_cast<double *>(points);
    else if (num_point > 0)
        RCHK(hipMemcpyAsync(d_pts, points, 16 * (size_t)num_point, hipMemcpyDefault, st), "upload");
    if (own_wt) d_wt = const_cast<double *>(weight);
    else if (num_point > 0)
        RCHK(hipMemcpyAsync(d_wt, weight, 8 * (size_t)num_point, hipMemcpyDefault, st), "upload");
    if (own_tri) d_tri = const_cast<int *>(triangle);
    else if (num_tri > 0)
        RCHK(hipMemcpyAsync(d_tri, triangle, 12 * (size_t)num_tri, hipMemcpyDefault, st), "upload");
    if (own_den) d_den = density;
    const dim3 gt((num_tri + 255) / 256), blk(256);
    launch_zero(st, d_status, zeroed);
    if (num_tri > 0)
        hipLaunchKernelGGL(k_tri_boxes, gt, blk, 0, st, d_pts, num_point, d_tri, num_tri, scale, n,
                           tiles_x, d_box, d_alw, d_count, d_status);
    launch_exclusive_scan(st, d_count, ntiles, d_start);
    MeshScratch more;
    int *host = mem.status();
    for (int round = 0; round < 2; ++round) {
        if (num_tri > 0)
            hipLaunchKernelGGL(k_tile_fill, gt, blk, 0, st, d_box, num_tri, tiles_x, d_start, d_cursor,
                               d_list, (int)cap, d_status);
        hipLaunchKernelGGL(k_raster, dim3((ntiles + 3) / 4), blk, 0, st, d_pts, d_wt, d_tri, d_list,
                           d_start, d_alw, tiles_x, ntiles, scale, n, d_den, d_status, host);
        RCHK(hipGetLastError(), "raster launch");
        RCHK(hipStreamSynchronize(st), "raster");
        if (host[0]) {
            mem.idle();
            return fail(CVT_ERR_ARG, "a triangle indexes a vertex outside [0, %d)", num_point);
        }
        if (!host[1]) break;
        if (host[2] < 0) {
            mem.idle();
            return fail(CVT_ERR_CAPACITY, "2^31 or more (triangle, tile) pairs");
        }
        cap = (size_t)host[2];
        RCHK(more.take(sizeof(int) * cap), "alloc");
        d_list = reinterpret_cast<int *>(more.base());
        RCHK(hipMemsetAsync(d_status + ST_OVERFLOW, 0, sizeof(int), st), "memset");
    }
    if (!own_den) {
        RCHK(hipMemcpyAsync(density, d_den, 4 * npx, hipMemcpyDefault, st), "download");
        RCHK(hipStreamSynchronize(st), "raster");
    }
    mem.idle();
    more.idle();
    return CVT_OK;
}

// ---------------------------------------------------------------------------
// cvt_rasterize_noalloc: cvt_rasterize for callers that cannot allocate.  All
// of its working memory (triangle boxes, the thin-triangle list, per-tile
// counts and list starts, the (triangle, tile) lists and the status words)
// lives in one static device array, so the call allocates nothing.  Each
// device holds its own copy of the array; its address is looked up once per
// device with hipGetSymbolAddress.  Every call on a device shares that
// device's array: calls that overlap on one device race.
// ---------------------------------------------------------------------------
namespace cvt {

#define NOALLOC_MAX_N 4096
#define NOALLOC_MAX_TRI (1 << 18)
#define NOALLOC_MAX_PAIRS (1 << 21)
#define NOALLOC_TILES ((NOALLOC_MAX_N / RT) * (NOALLOC_MAX_N / RT))

// byte offsets of the parts (each a multiple of 256)
enum : size_t {
    NA_BOX = 0,
    NA_ALW = NA_BOX + sizeof(TriBox) * (size_t)NOALLOC_MAX_TRI,
    NA_STATUS = NA_ALW + sizeof(int) * (size_t)NOALLOC_MAX_TRI,
    NA_COUNT = NA_STATUS + 256,
    NA_CURSOR = NA_COUNT + sizeof(int) * (size_t)NOALLOC_TILES,
    NA_START = NA_CURSOR + sizeof(int) * (size_t)NOALLOC_TILES,
    NA_LIST = NA_START + sizeof(int) * ((size_t)NOALLOC_TILES + 64),
    NA_BYTES = NA_LIST + sizeof(int) * (size_t)NOALLOC_MAX_PAIRS,
};
static_assert(NA_ALW % 256 == 0 && NA_STATUS % 256 == 0 && NA_COUNT % 256 == 0 &&
                  NA_CURSOR % 256 == 0 && NA_START % 256 == 0 && NA_LIST % 256 == 0,
              "scratch parts must stay 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[NA_BYTES];

#define NOALLOC_MAX_DEVICES 64
static unsigned char *g_scratch_ptr[NOALLOC_MAX_DEVICES];

// the device address of this device's scratch (looked up on its first use)
static int scratch_of(int dev, unsigned char **out)
{
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
        return fail(CVT_ERR_ARG, "device %d beyond the %d the no-alloc path supports", dev,
                    NOALLOC_MAX_DEVICES);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(CVT_ERR_HIP, "scratch address: %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch_ptr[dev];
    return CVT_OK;
}

static __global__ void k_zero_i32(int *__restrict__ p, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x)
        p[i] = 0;
}

// true when p is memory the device can read and write (device, pinned or
// managed memory); pageable host memory is not
static bool device_accessible(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.devicePointer != nullptr;
}

}  // namespace cvt

extern "C" int cvt_rasterize_noalloc(const double *points, const double *weight, int num_point,
                                     const int *triangle, int num_tri, float *density,
                                     double scale, int n)
{
    clear_error();
    if (n < 1 || n > NOALLOC_MAX_N)
        return fail(CVT_ERR_ARG, "n = %d outside [1, %d] (the no-alloc limit)", n, NOALLOC_MAX_N);
    if (num_point < 0 || num_tri < 0) return fail(CVT_ERR_ARG, "negative sizes");
    if (num_tri > NOALLOC_MAX_TRI)
        return fail(CVT_ERR_ARG, "%d triangles above the no-alloc limit %d", num_tri,
                    NOALLOC_MAX_TRI);
    if (!density || (num_point > 0 && (!points || !weight)) || (num_tri > 0 && !triangle))
        return fail(CVT_ERR_ARG, "null array");
    if (!(scale > 0.0) || !isfinite(scale)) return fail(CVT_ERR_ARG, "scale %g", scale);
    if (!device_accessible(density) ||
        (num_point > 0 && (!device_accessible(points) || !device_accessible(weight))) ||
        (num_tri > 0 && !device_accessible(triangle)))
        return fail(CVT_ERR_ARG, "the no-alloc rasterizer needs device-accessible buffers");
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail(CVT_ERR_HIP, "no current device");
    unsigned char *base = nullptr;
    int rc = scratch_of(dev, &base);
    if (rc) return rc;
    TriBox *box = reinterpret_cast<TriBox *>(base + NA_BOX);
    int *alw = reinterpret_cast<int *>(base + NA_ALW);
    int *count = reinterpret_cast<int *>(base + NA_COUNT);
    int *cursor = reinterpret_cast<int *>(base + NA_CURSOR);
    int *start = reinterpret_cast<int *>(base + NA_START);
    int *list = reinterpret_cast<int *>(base + NA_LIST);
    int *status = reinterpret_cast<int *>(base + NA_STATUS);
    const int tiles_x = (n + RT - 1) / RT, ntiles = tiles_x * tiles_x;
    hipStream_t st = nullptr;   // the legacy default stream, as cvt_rasterize
    // the counts, cursors and status words left by the last call start at zero
    hipLaunchKernelGGL(k_zero_i32, dim3(256), dim3(256), 0, st, count, (long)ntiles);
    hipLaunchKernelGGL(k_zero_i32, dim3(256), dim3(256), 0, st, cursor, (long)ntiles);
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(64), 0, st, status, (long)ST_WORDS);
    if (num_tri > 0)
        hipLaunchKernelGGL(k_tri_boxes, dim3((num_tri + 255) / 256), dim3(256), 0, st, points,
                           num_point, triangle, num_tri, scale, n, tiles_x, box, alw, count, status);
    launch_exclusive_scan(st, count, ntiles, start);
    if (num_tri > 0)
        hipLaunchKernelGGL(k_tile_fill, dim3((num_tri + 255) / 256), dim3(256), 0, st, box,
                           num_tri, tiles_x, start, cursor, list, NOALLOC_MAX_PAIRS, status);
    hipLaunchKernelGGL(k_raster, dim3((ntiles + 3) / 4), dim3(256), 0, st, points, weight, triangle,
                       list, start, alw, tiles_x, ntiles, scale, n, density, status, nullptr);
    int h[3] = {0, 0, 0};
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(h, status, sizeof h, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return fail(CVT_ERR_HIP, "no-alloc raster: %s", hipGetErrorString(e));
    if (h[0]) return fail(CVT_ERR_ARG, "a triangle indexes a vertex outside [0, %d)", num_point);
    if (h[1])
        return fail(CVT_ERR_CAPACITY, "more than %d (triangle, tile) pairs (the no-alloc limit)",
                    NOALLOC_MAX_PAIRS);
    return CVT_OK;
}

