// mesh_scratch.h -- working memory and argument handling of the mesh calls
// (cvt_rasterize, cvt_locate_points, cvt_vertex_weights), which are complete
// in themselves: they hold no context, run on the legacy default stream and
// return when their results are written.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace cvt {

constexpr int kStatusWords = 16;

// One call's device memory and a few pinned words for the results the host
// reads.  Blocks go back to a small store on release, so that a call on a mesh
// like the last one's neither allocates nor frees.  With the lists' size read
// back between two halves of a call and each argument copied first, that was
// 245 us to locate 49152 points in an 11858-face mesh and 400 us for its vertex
// weights and 2048^2 raster, for 60 and 130 us of kernels; now 72 and 154 us.
// A block belongs to one call at a time, whatever thread makes it, and is
// released only after the call has waited for its work.  A block that a reset
// of the device has freed since is left alone.  The store holds the newest
// blocks, at most kScratchBlocks and kScratchBytes bytes per device; larger
// ones are freed at once, and all of them when a device allocation here fails or
// cvt_release_scratch is called.
constexpr int kScratchBlocks = 4;
constexpr size_t kScratchBytes = (size_t)64 << 20;

class MeshScratch {
public:
    MeshScratch() = default;
    ~MeshScratch();
    MeshScratch(const MeshScratch &) = delete;
    MeshScratch &operator=(const MeshScratch &) = delete;
    // device memory of at least `bytes` (once per object)
    hipError_t take(size_t bytes);
    // the call has waited for all its work (release waits otherwise)
    void idle() { idle_ = true; }
    char *base() const { return dev_; }
    size_t bytes() const { return bytes_; }
    int *status() const { return pinned_; }        // kStatusWords pinned ints

private:
    int device_ = -1;
    char *dev_ = nullptr;
    size_t bytes_ = 0;
    int *pinned_ = nullptr;
    bool idle_ = false;
};

void release_scratch();

// whether a kernel on the current device can take the argument as it is:
// device memory of that device, aligned for its type (anything else is copied)
bool in_place(const void *p, size_t align);
// whether two ranges meet
inline bool overlap(const void *a, size_t na, const void *b, size_t nb)
{
    const char *x = static_cast<const char *>(a), *y = static_cast<const char *>(b);
    return x && y && na && nb && x < y + nb && y < x + na;
}

// zeroes `bytes` (a multiple of 16) at p, 16-byte aligned, with one launch (a
// memset of a size that is no power of two takes two)
void launch_zero(hipStream_t st, void *p, size_t bytes);

// Whether the barycentric weights n2 / den, n3 / den and 1 - n2 / den - n3 / den,
// as they round, are all >= 0: 1 yes, 0 no, -1 take the divisions.  With den in
// (1e-150, 1e150), n < -1e-150 gives a negative quotient for certain and n >= 0
// one that is not, and 1e-7 den is far more than the quotients round by.  Of
// 4 million pixels of an ordinary mesh almost none needs the divisions, which
// every lane of a wave would wait for.
__device__ __forceinline__ int inside_sign(double n2, double n3, double den)
{
    if (!(den > 1e-150 && den < 1e150)) return -1;
    const double s = n2 + n3;
    if (n2 < -1e-150 || n3 < -1e-150 || s > 1.0000001 * den) return 0;
    return (n2 >= 0 && n3 >= 0 && s <= 0.9999999 * den) ? 1 : -1;
}
__device__ __forceinline__ bool inside_exact(double n2, double n3, double den)
{
    const double b2 = n2 / den, b3 = n3 / den, b1 = 1.0 - b2 - b3;
    return !(b1 < 0 || b2 < 0 || b3 < 0);
}

// Adds the (face, cell) pairs of a wave's lanes, at most 2^20 each, to a
// call's total; called by every lane of the wave.  The lists' starts are 32-bit
// sums, which wrap beyond 2^31 - 1 pairs: whether the lists hold all pairs is
// decided from this total.
__device__ __forceinline__ void add_pairs(int pairs, unsigned long long *total)
{
    for (int o = 32; o > 0; o >>= 1) pairs += __shfl_xor(pairs, o, 64);
    if ((threadIdx.x & 63) == 0 && pairs > 0) atomicAdd(total, (unsigned long long)pairs);
}
// the total as the host reads it: -1 where no list of 32-bit starts holds it
__device__ __forceinline__ int pairs_word(unsigned long long total)
{
    return total > 0x7fffffffull ? -1 : (int)total;
}

// positions of a call's buffers in its scratch, each at a 256-byte boundary:
// run once to size it and once to place them
struct Carver {
    char *base = nullptr;
    size_t at = 0;
    template <typename T>
    void operator()(T *&p, size_t n)
    {
        at = (at + 255) & ~(size_t)255;
        p = reinterpret_cast<T *>(base + at);
        at += n * sizeof(T);
    }
};

}  // namespace cvt
