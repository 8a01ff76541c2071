// locate.hip -- point location in a 2D triangle mesh (replaces the brute-force
// face scan of the reference's recover(), source/recover.h:63-81, run for
// every site at :109-125 and for every output triangle's centroid at
// :134-141).
//
// Rule (the reference's locate(), source/recover.h:63-81): a point lies in the
// first face, in face order, whose three float64 barycentric weights (the
// formula of source/recover.h:30-53) are all >= 0; a face with a zero
// denominator never holds a point.  The weights are returned in the face's
// vertex order: vertex 0 gets 1 - w1 - w2, vertices 1 and 2 get w1 and w2
// (source/recover.h:79, the argument order of barycentric()).  The 3D point
// of a located site is sum_j w_j * P3[v_j], summed in that order from 0.0
// (source/recover.h:117-123).  A non-finite query point is in no face (the
// reference would accept it in the first non-degenerate face: NaN weights
// fail no "< 0" test).
//
// Instead of testing every face for every point (O(Q F)), faces are binned
// into a G x G grid over the vertices' bounding box by a conservative box (a
// counting sort: count, prefix sum, fill; linear in the number of (face, bin)
// pairs).  A point tests the faces of its bin and keeps the lowest-index hit,
// which is the first hit in face order: every face holding the point lists
// it in that bin.  Faces so thin that rounding could accept points well
// outside their box go to an "always" list that every point tests.
// Contraction is off for this file: every expression rounds as written, as
// in the oracle.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/cvt.h"
#include "cvt_engine.h"
#include "mesh_scratch.h"
#include "scan.h"

namespace cvt {

struct FaceBox {
    int x0, x1, y0, y1;   // inclusive bin range; x0 > x1 = in no bin
};

// the bin grid: G x G bins over [ox, ox + G / inv) x [oy, oy + G / inv)
struct BinGrid {
    double ox, oy, inv;
    int G;
};

// a double as an unsigned key in the same order (NaN excluded), never 0
__device__ __forceinline__ unsigned long long order_key(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : b | (1ull << 63);
}
__device__ __forceinline__ double from_key(unsigned long long k)
{
    return __longlong_as_double((long long)((k >> 63) ? k & ~(1ull << 63) : ~k));
}

// square bins over the vertex box (no vertex, a zero-size or a non-finite
// box: one bin).  bb: the largest keys of -x, -y (as complements), x and y,
// 0 where no vertex had one.
__device__ __forceinline__ BinGrid bin_grid(const unsigned long long *__restrict__ bb, int G)
{
    BinGrid g;
    const double x0 = bb[0] ? from_key(~bb[0]) : INFINITY, y0 = bb[1] ? from_key(~bb[1]) : INFINITY;
    const double x1 = bb[2] ? from_key(bb[2]) : -INFINITY, y1 = bb[3] ? from_key(bb[3]) : -INFINITY;
    const double ex = x1 - x0, ey = y1 - y0, ext = ex < ey ? ey : ex;
    g.ox = isfinite(x0) ? x0 : 0.0;
    g.oy = isfinite(y0) ? y0 : 0.0;
    g.inv = (ext > 0.0 && isfinite(ext)) ? (double)G / ext : 0.0;
    g.G = g.inv == 0.0 ? 1 : G;
    return g;
}

// bin of a coordinate: monotone in v (so a point inside a box maps inside the
// box's bin range) and clamped to the grid, NaN to bin 0
__device__ __forceinline__ int bin_of(double v, double o, double inv, int G)
{
    double t = (v - o) * inv;
    t = fmax(0.0, fmin(t, (double)(G - 1)));
    return (int)floor(t);
}

// bounding box of the vertices as order keys (bb zeroed by the caller)
__global__ __launch_bounds__(256) void k_vertex_bounds(const double *__restrict__ uv, int nv,
                                                       unsigned long long *__restrict__ bb)
{
    __shared__ double r[4][4];
    double m[4] = {INFINITY, INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nv; i += gridDim.x * 256) {
        const double x = uv[2 * i], y = uv[2 * i + 1];
        m[0] = fmin(m[0], x); m[1] = fmin(m[1], y); m[2] = fmax(m[2], x); m[3] = fmax(m[3], y);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        for (int o = 32; o > 0; o >>= 1) {
            const double v = __shfl_xor(m[c], o, 64);
            m[c] = c < 2 ? fmin(m[c], v) : fmax(m[c], v);
        }
        if ((threadIdx.x & 63) == 0) r[c][threadIdx.x >> 6] = m[c];
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= 4) return;
    const double lo = fmin(fmin(r[c][0], r[c][1]), fmin(r[c][2], r[c][3]));
    const double hi = fmax(fmax(r[c][0], r[c][1]), fmax(r[c][2], r[c][3]));
    atomicMax(&bb[c], c < 2 ? ~order_key(lo) : order_key(hi));
}

// the corners of a face, in one 48-byte record: a query reads a candidate
// face with one gather behind its list entry
struct FaceXY {
    double x1, y1, x2, y2, x3, y3;
};

// status: {a face indexes outside, pairs beyond the list, faces in alw, -, and
// the (face, bin) pairs in 64 bits}
constexpr int kStatus = 8;
__device__ __forceinline__ unsigned long long *pair_total(int *status)
{
    return reinterpret_cast<unsigned long long *>(status + 4);
}

// face i: index validation, the corner record and the conservative bin box.
// Faces to test everywhere are appended to alw in any order (a query keeps the
// lowest-index hit).
__device__ __forceinline__ FaceBox face_box(const double *__restrict__ uv, int nv,
                                            const int *__restrict__ tri, int i, const BinGrid &g,
                                            FaceXY *__restrict__ xy, int *__restrict__ alw,
                                            int *__restrict__ status)
{
    const int a = tri[3 * i], b = tri[3 * i + 1], c = tri[3 * i + 2];
    FaceBox bx = {1, 0, 1, 0};
    if ((unsigned)a >= (unsigned)nv || (unsigned)b >= (unsigned)nv || (unsigned)c >= (unsigned)nv) {
        status[0] = 1;
        return bx;
    }
    const double x1 = uv[2 * a], y1 = uv[2 * a + 1];
    const double x2 = uv[2 * b], y2 = uv[2 * b + 1];
    const double x3 = uv[2 * c], y3 = uv[2 * c + 1];
    xy[i] = FaceXY{x1, y1, x2, y2, x3, y3};
    const double v0x = x2 - x1, v0y = y2 - y1, v1x = x3 - x1, v1y = y3 - y1;
    const double d00 = v0x * v0x + v0y * v0y, d11 = v1x * v1x + v1y * v1y;
    const double d01 = v0x * v1x + v0y * v1y;
    const double den = d00 * d11 - d01 * d01;
    if (den == 0) return bx;                         // holds no point
    if (!(den > 1e-12 * d00 * d11)) {                // thin or non-finite: test everywhere
        alw[atomicAdd(&status[2], 1)] = i;
        return bx;
    }
    const double xmin = fmin(x1, fmin(x2, x3)), xmax = fmax(x1, fmax(x2, x3));
    const double ymin = fmin(y1, fmin(y2, y3)), ymax = fmax(y1, fmax(y2, y3));
    const double eps = 1e-9 * fmax(xmax - xmin, ymax - ymin) + 1e-300;
    bx.x0 = bin_of(xmin - eps, g.ox, g.inv, g.G);
    bx.x1 = bin_of(xmax + eps, g.ox, g.inv, g.G);
    bx.y0 = bin_of(ymin - eps, g.oy, g.inv, g.G);
    bx.y1 = bin_of(ymax + eps, g.oy, g.inv, g.G);
    return bx;
}

// per face: its record and box, and its (face, bin) pairs counted per bin and
// in all
__global__ void k_face_boxes(const double *__restrict__ uv, int nv, const int *__restrict__ tri,
                             int nf, const unsigned long long *__restrict__ bb, int G,
                             FaceXY *__restrict__ xy, FaceBox *__restrict__ box,
                             int *__restrict__ alw, int *__restrict__ count,
                             int *__restrict__ status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int pairs = 0;
    if (i < nf) {
        const BinGrid g = bin_grid(bb, G);
        const FaceBox bx = face_box(uv, nv, tri, i, g, xy, alw, status);
        box[i] = bx;
        for (int y = bx.y0; y <= bx.y1; ++y)
            for (int x = bx.x0; x <= bx.x1; ++x) atomicAdd(&count[y * g.G + x], 1);
        pairs = (bx.x1 - bx.x0 + 1) * (bx.y1 - bx.y0 + 1);
    }
    add_pairs(pairs, pair_total(status));
}

// (face, bin) pairs: each face writes its index into the lists of its bins;
// with more pairs than the list holds, nothing but the flag
__global__ void k_bin_fill(const FaceBox *__restrict__ box, int nf,
                           const unsigned long long *__restrict__ bb, int grid,
                           const int *__restrict__ start, int *__restrict__ cursor,
                           int *__restrict__ list, int cap, int *__restrict__ status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nf) return;
    if (*pair_total(status) > (unsigned long long)cap) {
        if (i == 0) status[1] = 1;
        return;
    }
    const FaceBox b = box[i];
    if (b.x0 > b.x1) return;
    const int G = bin_grid(bb, grid).G;
    for (int y = b.y0; y <= b.y1; ++y)
        for (int x = b.x0; x <= b.x1; ++x) {
            const int bin = y * G + x;
            list[start[bin] + atomicAdd(&cursor[bin], 1)] = i;
        }
}

// one thread per query point: the lowest-index face of its bin list and of
// the "always" list that holds it; face -1 when none does.  Candidates are
// decided by the signs of the weights' numerators, and the weights divided
// out once, for the hit.  kAtOnce candidates are read together.  host, pinned,
// receives the status and the number of pairs.
// Bound by the latency of list entry -> face record: 49152 points in an
// 11858-face mesh 13 us (17 us with indices and corners as separate gathers
// and two divisions per candidate; 15 us with eight at a time).
constexpr int kAtOnce = 4;
__global__ __launch_bounds__(256) void k_locate(const FaceXY *__restrict__ xy,
                                                const double *__restrict__ p3,
                                                const int *__restrict__ tri,
                                                const int *__restrict__ list,
                                                const int *__restrict__ start,
                                                const int *__restrict__ alw,
                                                const unsigned long long *__restrict__ bb, int G,
                                                const double *__restrict__ q, int nq,
                                                int *__restrict__ face, double *__restrict__ w,
                                                double *__restrict__ out3,
                                                int *__restrict__ status, int *__restrict__ host)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {
        host[0] = status[0];
        host[1] = status[1];
        host[2] = pairs_word(*pair_total(status));
    }
    if (k >= nq || status[0] || status[1]) return;
    const int nalw = status[2];
    const double x = q[2 * k], y = q[2 * k + 1];
    int hit = -1;
    double h1 = 0.0, h2 = 0.0, hd = 1.0;
    // a non-finite point is in no face
    if (isfinite(x) && isfinite(y)) {
        const BinGrid g = bin_grid(bb, G);
        const int bin = bin_of(y, g.oy, g.inv, g.G) * g.G + bin_of(x, g.ox, g.inv, g.G);
        const int a = start[bin], n = start[bin + 1] - a;
        for (int j0 = 0; j0 < n + nalw; j0 += kAtOnce) {
            int id[kAtOnce];
            FaceXY f[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                const int j = min(j0 + u, n + nalw - 1);
                id[u] = (j < n) ? list[a + j] : alw[j - n];
            }
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) f[u] = xy[id[u]];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                // a lower-index hit is known (or the list ended: its last again)
                if (hit >= 0 && id[u] >= hit) continue;
                const double v0x = f[u].x2 - f[u].x1, v0y = f[u].y2 - f[u].y1;
                const double v1x = f[u].x3 - f[u].x1, v1y = f[u].y3 - f[u].y1;
                const double v2x = x - f[u].x1, v2y = y - f[u].y1;
                const double d00 = v0x * v0x + v0y * v0y;
                const double d01 = v0x * v1x + v0y * v1y;
                const double d11 = v1x * v1x + v1y * v1y;
                const double d20 = v2x * v0x + v2y * v0y;
                const double d21 = v2x * v1x + v2y * v1y;
                const double den = d00 * d11 - d01 * d01;
                const double n1 = d11 * d20 - d01 * d21, n2 = d00 * d21 - d01 * d20;
                if (den == 0) continue;
                const int in = inside_sign(n1, n2, den);
                if (in == 0 || (in < 0 && !inside_exact(n1, n2, den))) continue;
                hit = id[u];
                h1 = n1; h2 = n2; hd = den;
            }
        }
    }
    double w0 = -1, w1 = -1, w2 = -1;
    if (hit >= 0) {
        w1 = h1 / hd;
        w2 = h2 / hd;
        w0 = 1.0 - w1 - w2;
    }
    face[k] = hit;
    if (w) {
        w[3 * k] = w0;
        w[3 * k + 1] = w1;
        w[3 * k + 2] = w2;
    }
    if (out3) {
        double r[3] = {0.0, 0.0, 0.0};
        if (hit >= 0) {
            const int v[3] = {tri[3 * hit], tri[3 * hit + 1], tri[3 * hit + 2]};
            const double wt[3] = {w0, w1, w2};
            for (int c = 0; c < 3; ++c)
                for (int j = 0; j < 3; ++j) r[c] += p3[3 * v[j] + c] * wt[j];
        }
        out3[3 * k] = r[0];
        out3[3 * k + 1] = r[1];
        out3[3 * k + 2] = r[2];
    }
}

__global__ __launch_bounds__(256) void k_zero(uint4 *__restrict__ p, long n)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = make_uint4(0, 0, 0, 0);
}

void launch_zero(hipStream_t st, void *p, size_t bytes)
{
    const long n = (long)(bytes / 16);
    if (n > 0)
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                           static_cast<uint4 *>(p), n);
}

void launch_exclusive_scan(hipStream_t st, const int *count, int n, int *start)
{
    launch_scan(st, CountLoad{count}, n, start, ScanDone());
}

}  // namespace cvt

using namespace cvt;

#define LCHK(call, what)                                                                  \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess) return fail(CVT_ERR_HIP, "%s: %s", what, hipGetErrorString(e_)); \
    } while (0)

// One pass over the mesh and one over the queries, with one wait at the end:
// the bin grid stays on the device, and the lists get room for the pairs of
// an ordinary mesh (four to six per face); a mesh with more (long, slanted
// faces) is seen at the wait, and its lists are filled again with room for
// all.  Arguments in memory of the device are used where they are.
extern "C" int cvt_locate_points(const double *uv, const double *p3, int nv, const int *tri,
                                 int nf, const double *q, int nq, int *face, double *w,
                                 double *out3)
{
    clear_error();
    if (nv < 0 || nf < 0 || nq < 0) return fail(CVT_ERR_ARG, "negative sizes");
    if ((nv > 0 && !uv) || (nf > 0 && !tri) || (nq > 0 && (!q || !face)))
        return fail(CVT_ERR_ARG, "null array");
    if (out3 && nv > 0 && !p3) return fail(CVT_ERR_ARG, "out3 needs the 3D vertices p3");
    if (nq == 0) return CVT_OK;
    // about two faces per bin, at most 1024 x 1024 bins
    const int G = std::max(1, std::min(1024, (int)ceil(sqrt((double)std::max(nf, 1) / 2.0))));
    hipStream_t st = nullptr;   // the legacy default stream, as the reference's calls use
    const size_t nva = (size_t)std::max(nv, 1), nfa = (size_t)std::max(nf, 1), nb = (size_t)G * G;
    const size_t n1 = (size_t)nq, b_uv = 16 * nva, b_tri = 12 * nfa, b_q = 16 * n1, b_p3 = 24 * nva;
    // outputs written in place must not meet an input, or one copied before
    auto clear_of = [&](const void *o, size_t bytes) {
        return !overlap(o, bytes, uv, b_uv) && !overlap(o, bytes, tri, b_tri) &&
               !overlap(o, bytes, q, b_q) && !(out3 && overlap(o, bytes, p3, b_p3));
    };
    const bool own_uv = nv > 0 && in_place(uv, 8), own_tri = nf > 0 && in_place(tri, 4);
    const bool own_q = in_place(q, 8), own_p3 = out3 && nv > 0 && in_place(p3, 8);
    const bool own_face = in_place(face, 4) && clear_of(face, 4 * n1);
    const bool own_w = w && in_place(w, 8) && clear_of(w, 24 * n1) && !overlap(w, 24 * n1, face, 4 * n1);
    const bool own_out3 = out3 && in_place(out3, 8) && clear_of(out3, 24 * n1) &&
                          !overlap(out3, 24 * n1, face, 4 * n1) && !overlap(out3, 24 * n1, w, 24 * n1);
    double *d_uv = nullptr, *d_p3 = nullptr, *d_q = nullptr, *d_w = nullptr, *d_out3 = nullptr;
    int *d_tri = nullptr, *d_list = nullptr, *d_count = nullptr, *d_cursor = nullptr,
        *d_start = nullptr, *d_alw = nullptr, *d_status = nullptr, *d_face = nullptr;
    unsigned long long *d_bb = nullptr;
    FaceBox *d_box = nullptr;
    FaceXY *d_xy = nullptr;
    size_t cap = std::min<size_t>(8 * nfa + 1024, INT32_MAX);
    MeshScratch mem;
    Carver carve;
    size_t zeroed = 0;
    auto layout = [&]() {
        carve.base = mem.base();
        carve.at = 0;
        carve(d_bb, 4);                          // zeroed from here
        carve(d_status, kStatus); carve(d_count, nb); carve(d_cursor, nb);
        zeroed = (carve.at + 255) & ~(size_t)255;
        carve(d_start, nb + 1); carve(d_box, nfa); carve(d_xy, nfa); carve(d_alw, nfa);
        if (!own_uv) carve(d_uv, 2 * nva);
        if (!own_tri) carve(d_tri, 3 * nfa);
        if (!own_q) carve(d_q, 2 * n1);
        if (!own_face) carve(d_face, n1);
        if (w && !own_w) carve(d_w, 3 * n1);
        if (out3 && !own_out3) carve(d_out3, 3 * n1);
        if (out3 && !own_p3) carve(d_p3, 3 * nva);
        carve(d_list, cap);
    };
    layout();
    LCHK(mem.take(carve.at), "alloc");
    layout();
    if (own_uv) d_uv = const_cast<double *>(uv);
    else if (nv > 0) LCHK(hipMemcpyAsync(d_uv, uv, 16 * (size_t)nv, hipMemcpyDefault, st), "upload");
    if (own_tri) d_tri = const_cast<int *>(tri);
    else if (nf > 0) LCHK(hipMemcpyAsync(d_tri, tri, 12 * (size_t)nf, hipMemcpyDefault, st), "upload");
    if (own_q) d_q = const_cast<double *>(q);
    else LCHK(hipMemcpyAsync(d_q, q, b_q, hipMemcpyDefault, st), "upload");
    if (own_p3) d_p3 = const_cast<double *>(p3);
    else if (out3 && nv > 0)
        LCHK(hipMemcpyAsync(d_p3, p3, 24 * (size_t)nv, hipMemcpyDefault, st), "upload");
    if (own_face) d_face = face;
    if (own_w) d_w = w;
    if (own_out3) d_out3 = out3;
    const dim3 gf((nf + 255) / 256), blk(256);
    launch_zero(st, d_bb, zeroed);
    if (nv > 0)
        hipLaunchKernelGGL(k_vertex_bounds, dim3(std::min(64, (nv + 255) / 256)), blk, 0, st, d_uv,
                           nv, d_bb);
    if (nf > 0)
        hipLaunchKernelGGL(k_face_boxes, gf, blk, 0, st, d_uv, nv, d_tri, nf, d_bb, G, d_xy, d_box,
                           d_alw, d_count, d_status);
    launch_exclusive_scan(st, d_count, (int)nb, d_start);
    MeshScratch more;
    int *host = mem.status();
    for (int round = 0; round < 2; ++round) {
        if (nf > 0)
            hipLaunchKernelGGL(k_bin_fill, gf, blk, 0, st, d_box, nf, d_bb, G, d_start, d_cursor,
                               d_list, (int)cap, d_status);
        hipLaunchKernelGGL(k_locate, dim3((nq + 255) / 256), blk, 0, st, d_xy, d_p3, d_tri, d_list,
                           d_start, d_alw, d_bb, G, d_q, nq, d_face, d_w, d_out3, d_status, host);
        LCHK(hipGetLastError(), "locate launch");
        LCHK(hipStreamSynchronize(st), "locate");
        if (host[0]) {
            mem.idle();
            return fail(CVT_ERR_ARG, "a face indexes a vertex outside [0, %d)", nv);
        }
        if (!host[1]) break;
        if (host[2] < 0) {
            mem.idle();
            return fail(CVT_ERR_CAPACITY, "2^31 or more (face, bin) pairs");
        }
        cap = (size_t)host[2];
        LCHK(more.take(sizeof(int) * cap), "alloc");
        d_list = reinterpret_cast<int *>(more.base());
        LCHK(hipMemsetAsync(d_status + 1, 0, sizeof(int), st), "reset");
    }
    if (!own_face) LCHK(hipMemcpyAsync(face, d_face, 4 * n1, hipMemcpyDefault, st), "download");
    if (w && !own_w) LCHK(hipMemcpyAsync(w, d_w, 24 * n1, hipMemcpyDefault, st), "download");
    if (out3 && !own_out3)
        LCHK(hipMemcpyAsync(out3, d_out3, 24 * n1, hipMemcpyDefault, st), "download");
    if (!own_face || (w && !own_w) || (out3 && !own_out3)) LCHK(hipStreamSynchronize(st), "locate");
    mem.idle();
    more.idle();
    return CVT_OK;
}
