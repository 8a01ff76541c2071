// scan.h -- exclusive prefix sums over a device array (or what a functor makes
// of one).
#pragma once

#include <hip/hip_runtime.h>

namespace cvt {

// Exclusive prefix sum of n counts into start[0 .. n] (both 16-byte aligned)
// over tiles of 4096 counts (1024 threads x 4 consecutive counts).  A count
// comes from load(base, n), the four from `base` (a multiple of 4; 0 past n),
// and done(total) runs in the workgroup that knows the sum, with all of its
// 1024 threads.  Up to Load::kOne counts one workgroup does it, a thread taking
// up to 32 consecutive counts whose loads are in flight together (k_scan_one);
// beyond that in three launches:
//   k_scan_tiles        each tile's total, parked in start[tile * 4096];
//   k_scan_tile_totals  one workgroup turns the parked totals into the tiles'
//                       offsets in place and writes start[n];
//   k_scan_apply        each tile reads its offset, then writes its starts
//                       (its first entry, the parked offset, last).
// The single workgroup is bound by the lines its strided loads fetch, so the
// line between the two depends on the width of what is loaded.  us behind the
// kernel that writes it, gaps included, one workgroup / three launches:
//               8192        12000       16384        24576        32768
//   counts      2.7 / 7.5   3.1 / 7.6   3.7 / 7.5    6.8 / 7.5    8.7 / 7.6
//   64-bit bids 4.2 / 7.8   8.5 / 7.8   10.7 / 7.8   16.5 / 8.3   21.5 / 8.5
constexpr int kScanTile = 4096;

// exclusive prefix sum over a 1024-thread workgroup of one value per thread;
// total receives the workgroup's sum (lds: 32 ints)
__device__ __forceinline__ int wg_exclusive_scan(int v, int *lds, int &total)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    __syncthreads();                       // lds is free (a previous call has read it)
    if (lane == 63) lds[wv] = x;
    __syncthreads();
    if (wv == 0) {
        int t = (lane < 16) ? lds[lane] : 0;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int y = __shfl_up(t, o, 64);
            if (lane >= o) t += y;
        }
        if (lane < 16) lds[16 + lane] = t;
    }
    __syncthreads();
    total = lds[31];
    return (wv > 0 ? lds[15 + wv] : 0) + x - v;
}

struct CountLoad {
    static constexpr int kOne = 24576;
    const int *count;
    __device__ __forceinline__ int4 operator()(long base, int n) const
    {
        if (base + 3 < n) return *reinterpret_cast<const int4 *>(count + base);
        int4 c = {0, 0, 0, 0};
        if (base < n) c.x = count[base];
        if (base + 1 < n) c.y = count[base + 1];
        if (base + 2 < n) c.z = count[base + 2];
        return c;
    }
};
struct ScanDone {
    __device__ __forceinline__ void operator()(int) const {}
};

template <class Load>
__global__ __launch_bounds__(1024) void k_scan_tiles(Load load, int n, int *__restrict__ start)
{
    __shared__ int lds[32];
    const long tile0 = (long)blockIdx.x * kScanTile;
    const int4 c = load(tile0 + 4 * threadIdx.x, n);
    int total;
    wg_exclusive_scan(c.x + c.y + c.z + c.w, lds, total);
    if (threadIdx.x == 0) start[tile0] = total;
}

template <class Done>
__global__ __launch_bounds__(1024) void k_scan_tile_totals(int *__restrict__ start, int n,
                                                           int ntiles, Done done)
{
    __shared__ int lds[32];
    int carry = 0;
    for (int c = 0; c < ntiles; c += 1024) {
        const int b = c + (int)threadIdx.x;
        const long at = (long)b * kScanTile;
        const int v = (b < ntiles) ? start[at] : 0;
        int total;
        const int ex = wg_exclusive_scan(v, lds, total);
        if (b < ntiles) start[at] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) start[n] = carry;
    done(carry);
}

template <class Load>
__global__ __launch_bounds__(1024) void k_scan_apply(Load load, int n, int *__restrict__ start)
{
    __shared__ int lds[32];
    const long tile0 = (long)blockIdx.x * kScanTile;
    const int off = start[tile0];          // read by every thread before the scan's barriers
    const long base = tile0 + 4 * threadIdx.x;
    const int4 c = load(base, n);
    int total;
    int run = off + wg_exclusive_scan(c.x + c.y + c.z + c.w, lds, total);
    const int v[4] = {c.x, c.y, c.z, c.w};
    for (int k = 0; k < 4; ++k)
        if (base + k < n) {
            start[base + k] = run;
            run += v[k];
        }
}

template <int QUADS, class Load, class Done>
__global__ __launch_bounds__(1024) void k_scan_one(Load load, int n, int *__restrict__ start,
                                                   Done done)
{
    __shared__ int lds[32];
    const long base = 4L * QUADS * threadIdx.x;
    int4 c[QUADS];
#pragma unroll
    for (int k = 0; k < QUADS; ++k) c[k] = load(base + 4 * k, n);
    int sum = 0;
#pragma unroll
    for (int k = 0; k < QUADS; ++k) sum += c[k].x + c[k].y + c[k].z + c[k].w;
    int total;
    int run = wg_exclusive_scan(sum, lds, total);
#pragma unroll
    for (int k = 0; k < QUADS; ++k) {
        const long at = base + 4 * k;
        const int4 s = {run, run + c[k].x, run + c[k].x + c[k].y, run + c[k].x + c[k].y + c[k].z};
        run = s.w + c[k].w;
        if (at + 3 < n) {
            *reinterpret_cast<int4 *>(start + at) = s;
            continue;
        }
        if (at < n) start[at] = s.x;
        if (at + 1 < n) start[at + 1] = s.y;
        if (at + 2 < n) start[at + 2] = s.z;
    }
    if (threadIdx.x == 0) start[n] = total;
    done(total);
}

template <class Load, class Done>
void launch_scan(hipStream_t st, Load load, int n, int *start, Done done)
{
    static_assert(Load::kOne <= 32768, "eight quads per thread");
    const dim3 b(1024);
#define CVT_SCAN_ONE(Q) \
    hipLaunchKernelGGL((k_scan_one<Q, Load, Done>), dim3(1), b, 0, st, load, n, start, done)
    if (n <= Load::kOne) {
        if (n <= 4096) CVT_SCAN_ONE(1);
        else if (Load::kOne <= 8192 || n <= 8192) CVT_SCAN_ONE(2);
        else if constexpr (Load::kOne > 8192) {
            if (n <= 16384) CVT_SCAN_ONE(4);
            else CVT_SCAN_ONE(8);
        }
#undef CVT_SCAN_ONE
        return;
    }
    const int ntiles = (int)(((long)n + kScanTile - 1) / kScanTile);
    hipLaunchKernelGGL((k_scan_tiles<Load>), dim3(ntiles), b, 0, st, load, n, start);
    hipLaunchKernelGGL((k_scan_tile_totals<Done>), dim3(1), b, 0, st, start, n, ntiles, done);
    hipLaunchKernelGGL((k_scan_apply<Load>), dim3(ntiles), b, 0, st, load, n, start);
}

}  // namespace cvt
