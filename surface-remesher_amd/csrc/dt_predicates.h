// dt_predicates.h -- exact orientation and in-circle signs for float64 points.
//
// Each predicate is evaluated in float64 first, with an error bound that
// decides whether the rounded sign is certain (the filter of Shewchuk's
// adaptive predicates, "Adaptive Precision Floating-Point Arithmetic and Fast
// Robust Geometric Predicates", 1997, with its first-stage bounds doubled).
// When it is not, the sign is computed exactly: every coordinate involved is
// written as m * 2^e with m an odd 53-bit integer and all of them are scaled
// to the smallest e among them, so that the determinant is an integer.  Its
// size is then known: the filter failed, so it is at most twice the filter's
// bound.  Where that is below 2^63 (2^127) units it is computed modulo 2^64
// (2^128) with wrapping arithmetic, whatever the size of its terms, and read
// as a signed number.  That takes one point's neighbourhood to some 2^27
// (2^43) units of the finest bit, which pixel lattices and float32 points
// meet; the wide evaluation that decides the rest took 10 to 15 us of a
// thread, which a degenerate input (a collinear boundary, a pixel lattice)
// spent in most passes.
// The rest is evaluated in fixed-width two's-complement integers (int128
// differences, 256-bit products, 512-bit in-circle terms), exact when the
// scaled coordinates fit in 124 bits, i.e. when the coordinates of one
// predicate span at most 2^71 units of their finest bit (any float32 input in
// pixel units does); otherwise the predicate reports a range error through
// *err and returns 0.
//
// The same source compiles for the host (g++) and for gfx950 (hipcc).  err,
// when not null, must point to global memory on the device.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define DT_HD __host__ __device__ inline
#define DT_HD_COLD __host__ __device__ inline __attribute__((noinline))
#else
#define DT_HD inline
#define DT_HD_COLD inline __attribute__((noinline))
#endif

namespace cvt {
namespace dt {

enum { DT_ERR_DEGENERATE = 1, DT_ERR_RANGE = 2, DT_ERR_CAPACITY = 4, DT_ERR_INPUT = 8,
       DT_ERR_CROSS = 16 };

typedef unsigned __int128 u128;
typedef __int128 i128;

// sets error bits; on the device err is global memory shared by all lanes
DT_HD void set_flag(int *err, int bits)
{
    if (!err) return;
#if defined(__HIP_DEVICE_COMPILE__)
    atomicOr(err, bits);
#else
    *err |= bits;
#endif
}

template <int N> struct Big {
    uint64_t w[N];                                  // two's complement, limb 0 lowest
};

template <int N> DT_HD Big<N> big_from(i128 v)
{
    Big<N> r;
    r.w[0] = (uint64_t)v;
    r.w[1] = (uint64_t)(v >> 64);
    const uint64_t ext = v < 0 ? ~0ull : 0ull;
    for (int i = 2; i < N; ++i) r.w[i] = ext;
    return r;
}

template <int N> DT_HD bool big_neg(const Big<N> &a) { return (a.w[N - 1] >> 63) != 0; }

template <int N> DT_HD Big<N> big_negate(const Big<N> &a)
{
    Big<N> r;
    uint64_t carry = 1;
    for (int i = 0; i < N; ++i) {
        const u128 s = (u128)(~a.w[i]) + carry;
        r.w[i] = (uint64_t)s;
        carry = (uint64_t)(s >> 64);
    }
    return r;
}

template <int N> DT_HD Big<N> big_add(const Big<N> &a, const Big<N> &b)
{
    Big<N> r;
    uint64_t carry = 0;
    for (int i = 0; i < N; ++i) {
        const u128 s = (u128)a.w[i] + b.w[i] + carry;
        r.w[i] = (uint64_t)s;
        carry = (uint64_t)(s >> 64);
    }
    return r;
}

template <int N> DT_HD Big<N> big_sub(const Big<N> &a, const Big<N> &b)
{
    return big_add(a, big_negate(b));
}

template <int N> DT_HD int big_sign(const Big<N> &a)
{
    if (big_neg(a)) return -1;
    for (int i = 0; i < N; ++i)
        if (a.w[i]) return 1;
    return 0;
}

// signed N-limb x signed N-limb -> 2N limbs (the caller keeps |a|, |b| small
// enough that the product fits 2N limbs with its sign)
template <int N> DT_HD Big<2 * N> big_mul(Big<N> a, Big<N> b)
{
    const bool na = big_neg(a), nb = big_neg(b);
    if (na) a = big_negate(a);
    if (nb) b = big_negate(b);
    Big<2 * N> r;
    for (int i = 0; i < 2 * N; ++i) r.w[i] = 0;
    for (int i = 0; i < N; ++i) {
        uint64_t carry = 0;
        for (int j = 0; j < N; ++j) {
            const u128 p = (u128)a.w[i] * b.w[j] + r.w[i + j] + carry;
            r.w[i + j] = (uint64_t)p;
            carry = (uint64_t)(p >> 64);
        }
        r.w[i + N] = carry;
    }
    return na != nb ? big_negate(r) : r;
}

// x = m * 2^e with m odd (or m = 0, e = 0)
struct Fx {
    int64_t m;
    int e;
};

DT_HD Fx decompose(double x)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const int be = (int)((u >> 52) & 0x7ff);
    uint64_t f = u & ((1ull << 52) - 1);
    int e;
    if (be == 0) {
        e = -1074;                                  // subnormal or zero
    } else {
        f |= 1ull << 52;
        e = be - 1075;
    }
    Fx r;
    if (f == 0) {
        r.m = 0;
        r.e = 0;
        return r;
    }
    const int tz = __builtin_ctzll(f);
    f >>= tz;
    r.m = (u >> 63) ? -(int64_t)f : (int64_t)f;
    r.e = e + tz;
    return r;
}

// scales k coordinates to integers at their common finest bit; false if one
// would need more than 124 bits
template <int K> DT_HD bool to_integers(const double (&x)[K], i128 (&X)[K])
{
    Fx f[K];
    int emin = 1 << 30;
    for (int i = 0; i < K; ++i) {
        f[i] = decompose(x[i]);
        if (f[i].m != 0 && f[i].e < emin) emin = f[i].e;
    }
    for (int i = 0; i < K; ++i) {
        if (f[i].m == 0) {
            X[i] = 0;
            continue;
        }
        const int s = f[i].e - emin;                // m has at most 53 bits
        if (s > 71) return false;
        X[i] = (i128)f[i].m * ((i128)1 << s);
    }
    return true;
}

// The lowest set bit of k coordinates as an exponent (0 when all are zero),
// and how far the lowest set bit of any of them lies above it (to_integers
// takes 71); false for inf and NaN.
template <int K> DT_HD bool finest_bit(const double (&x)[K], int &emin, int &span)
{
    emin = 1 << 30;
    int emax = -(1 << 30);
    for (int i = 0; i < K; ++i) {
        const uint64_t u = __builtin_bit_cast(uint64_t, x[i]);
        const int be = (int)((u >> 52) & 0x7ff);
        const uint64_t f = u & ((1ull << 52) - 1);
        if (be == 0x7ff) return false;
        if (be == 0 && f == 0) continue;
        const int e0 = be == 0 ? -1074 : be - 1075;
        const int e = f ? e0 + __builtin_ctzll(f) : e0 + 52;
        if (e < emin) emin = e;
        if (e > emax) emax = e;
    }
    if (emin == 1 << 30) emin = emax = 0;
    span = emax - emin;
    return true;
}

// x * 2^-emin modulo 2^64 / 2^128 (x a multiple of 2^emin)
template <typename U> DT_HD U scaled_mod(double x, int emin)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const int be = (int)((u >> 52) & 0x7ff);
    uint64_t f = u & ((1ull << 52) - 1);
    int s;
    if (be == 0) {
        s = -1074 - emin;
    } else {
        f |= 1ull << 52;
        s = be - 1075 - emin;
    }
    // s < 0 only drops zero bits: emin is at most the coordinate's lowest bit
    U v = s < 0 ? (U)(s > -64 ? f >> -s : 0) : s >= (int)(8 * sizeof(U)) ? (U)0 : (U)f << s;
    return (u >> 63) ? (U)0 - v : v;
}

// log2 of a positive finite normal v, rounded up
DT_HD int log2_up(double v)
{
    return (int)((__builtin_bit_cast(uint64_t, v) >> 52) & 0x7ff) - 1022;
}

template <typename U> DT_HD int sign_mod(U v)
{
    return v == 0 ? 0 : (v >> (8 * sizeof(U) - 1)) ? -1 : 1;
}

template <typename U> DT_HD int orient_mod(const double (&x)[6], int e)
{
    const U cx = scaled_mod<U>(x[4], e), cy = scaled_mod<U>(x[5], e);
    const U ax = scaled_mod<U>(x[0], e) - cx, ay = scaled_mod<U>(x[1], e) - cy;
    const U bx = scaled_mod<U>(x[2], e) - cx, by = scaled_mod<U>(x[3], e) - cy;
    return sign_mod<U>(ax * by - ay * bx);
}

template <typename U> DT_HD int incircle_mod(const double (&x)[8], int e)
{
    const U dx = scaled_mod<U>(x[6], e), dy = scaled_mod<U>(x[7], e);
    const U ax = scaled_mod<U>(x[0], e) - dx, ay = scaled_mod<U>(x[1], e) - dy;
    const U bx = scaled_mod<U>(x[2], e) - dx, by = scaled_mod<U>(x[3], e) - dy;
    const U cx = scaled_mod<U>(x[4], e) - dx, cy = scaled_mod<U>(x[5], e) - dy;
    return sign_mod<U>((ax * ax + ay * ay) * (bx * cy - cx * by) +
                       (bx * bx + by * by) * (cx * ay - ax * cy) +
                       (cx * cx + cy * cy) * (ax * by - bx * ay));
}

// the exact stages are rarely taken: kept out of line so that the callers'
// filters stay small
DT_HD_COLD int orient_wide(const double (&x)[6], int *err)
{
    i128 X[6];
    if (!to_integers<6>(x, X)) {
        set_flag(err, DT_ERR_RANGE);
        return 0;
    }
    const i128 acx = X[0] - X[4], acy = X[1] - X[5], bcx = X[2] - X[4], bcy = X[3] - X[5];
    const Big<4> l = big_mul<2>(big_from<2>(acx), big_from<2>(bcy));
    const Big<4> r = big_mul<2>(big_from<2>(acy), big_from<2>(bcx));
    return big_sign(big_sub(l, r));
}

// bound: the filter's, which the float determinant does not exceed (so the
// true one is below twice of it)
DT_HD_COLD int orient_exact(double ax, double ay, double bx, double by, double cx, double cy,
                            double bound, int *err)
{
    const double x[6] = {ax, ay, bx, by, cx, cy};
    int e, span;
    if (bound > 1e-290 && bound < 1e290 && finest_bit<6>(x, e, span)) {
        if (span > 71) {
            set_flag(err, DT_ERR_RANGE);
            return 0;
        }
        if (log2_up(bound) + 1 - 2 * e < 63) return orient_mod<uint64_t>(x, e);
    }
    return orient_wide(x, err);
}

// Whether the coordinates' highest bits are near enough that their lowest set
// bits, at most 52 below, lie within the 71 that to_integers takes: what is
// decided without the integer stages is left to them otherwise, which refuse a
// wider span.
template <int K> DT_HD bool near_exponents(const double (&x)[K])
{
    uint32_t lo = ~0u, hi = 0;
    for (int i = 0; i < K; ++i) {
        const uint32_t u = (uint32_t)(__builtin_bit_cast(uint64_t, x[i]) >> 32) & 0x7fffffffu;
        const uint32_t v = x[i] == 0.0 ? ~0u : u;
        hi = u > hi ? u : hi;
        lo = v < lo ? v : lo;
    }
    return lo == ~0u || (hi >> 20) - (lo >> 20) <= 19;
}

// whether a - b = d exactly (the rounding error of the difference is zero)
DT_HD bool exact_diff(double a, double b, double d)
{
    const double bv = a - d, av = d + bv;
    return (a - av) + (bv - b) == 0.0;
}

// The sign where all four differences are exact, as they are for neighbouring
// points and for points of one lattice: the rounded products decide when they
// differ (rounding is monotone), their errors otherwise.  Short enough to sit
// in line: collinear boundaries and lattice rows end here instead of in the
// integer stages, whose code a launch fetches anew (a triangle split on such a
// boundary took 12 us against 4.5 without).  2: undecided.
DT_HD int orient_products(double ax, double ay, double bx, double by, double cx, double cy,
                          double bound)
{
    const double u = ax - cx, v = by - cy, s = ay - cy, t = bx - cx;
    const double l = u * v, r = s * t;
    const double x[6] = {ax, ay, bx, by, cx, cy};
    if (!near_exponents<6>(x)) return 2;
    if (bound == 0.0 && (u == 0.0 || v == 0.0) && (s == 0.0 || t == 0.0)) return 0;
    if (!(bound > 1e-270 && bound < 1e270) || !exact_diff(ax, cx, u) || !exact_diff(by, cy, v) ||
        !exact_diff(ay, cy, s) || !exact_diff(bx, cx, t))
        return 2;
    const double d = l != r ? l - r : __builtin_fma(u, v, -l) - __builtin_fma(s, t, -r);
    return d > 0 ? 1 : d < 0 ? -1 : 0;
}

// sign of (a - c) x (b - c): > 0 when a, b, c turn counterclockwise
DT_HD int orient2d(double ax, double ay, double bx, double by, double cx, double cy, int *err)
{
    const double l = (ax - cx) * (by - cy);
    const double r = (ay - cy) * (bx - cx);
    const double det = l - r;
    const double bound = 6.7e-16 * (__builtin_fabs(l) + __builtin_fabs(r));
    // the bound holds away from underflow and overflow; NaN and inf fail the
    // comparisons and go to the exact stage, which decides or reports
    if ((det > bound || -det > bound) && bound > 1e-290 && bound < 1e290)
        return det > 0 ? 1 : -1;
    const int o = orient_products(ax, ay, bx, by, cx, cy, bound);
    return o != 2 ? o : orient_exact(ax, ay, bx, by, cx, cy, bound, err);
}

DT_HD_COLD int incircle_wide(const double (&x)[8], int *err)
{
    i128 X[8];
    if (!to_integers<8>(x, X)) {
        set_flag(err, DT_ERR_RANGE);
        return 0;
    }
    const i128 adx = X[0] - X[6], ady = X[1] - X[7];
    const i128 bdx = X[2] - X[6], bdy = X[3] - X[7];
    const i128 cdx = X[4] - X[6], cdy = X[5] - X[7];
    auto sq = [](i128 u, i128 v) {
        return big_add(big_mul<2>(big_from<2>(u), big_from<2>(u)),
                       big_mul<2>(big_from<2>(v), big_from<2>(v)));
    };
    auto cross = [](i128 u1, i128 v1, i128 u2, i128 v2) {   // u1 v2 - u2 v1
        return big_sub(big_mul<2>(big_from<2>(u1), big_from<2>(v2)),
                       big_mul<2>(big_from<2>(u2), big_from<2>(v1)));
    };
    const Big<4> al = sq(adx, ady), bl = sq(bdx, bdy), cl = sq(cdx, cdy);
    const Big<4> bc = cross(bdx, bdy, cdx, cdy), ca = cross(cdx, cdy, adx, ady),
                 ab = cross(adx, ady, bdx, bdy);
    const Big<8> det = big_add(big_add(big_mul<4>(al, bc), big_mul<4>(bl, ca)), big_mul<4>(cl, ab));
    return big_sign(det);
}

// bound as in orient_exact
DT_HD_COLD int incircle_exact(const double (&x)[8], double bound, int *err)
{
    int e, span;
    if (bound > 1e-290 && bound < 1e290 && finest_bit<8>(x, e, span)) {
        if (span > 71) {
            set_flag(err, DT_ERR_RANGE);
            return 0;
        }
        const int bits = log2_up(bound) + 1 - 4 * e;
        if (bits < 63) return incircle_mod<uint64_t>(x, e);
        if (bits < 127) return incircle_mod<u128>(x, e);
    }
    return incircle_wide(x, err);
}

// > 0 when d lies inside the circle through a, b, c (counterclockwise), < 0
// outside, 0 on it
DT_HD int incircle(double ax, double ay, double bx, double by, double cx, double cy, double dx,
                   double dy, int *err)
{
    const double adx = ax - dx, ady = ay - dy, bdx = bx - dx, bdy = by - dy;
    const double cdx = cx - dx, cdy = cy - dy;
    const double bdxcdy = bdx * cdy, cdxbdy = cdx * bdy;
    const double cdxady = cdx * ady, adxcdy = adx * cdy;
    const double adxbdy = adx * bdy, bdxady = bdx * ady;
    const double alift = adx * adx + ady * ady;
    const double blift = bdx * bdx + bdy * bdy;
    const double clift = cdx * cdx + cdy * cdy;
    const double det = alift * (bdxcdy - cdxbdy) + blift * (cdxady - adxcdy) +
                       clift * (adxbdy - bdxady);
    const double perm = (__builtin_fabs(bdxcdy) + __builtin_fabs(cdxbdy)) * alift +
                        (__builtin_fabs(cdxady) + __builtin_fabs(adxcdy)) * blift +
                        (__builtin_fabs(adxbdy) + __builtin_fabs(bdxady)) * clift;
    const double bound = 2.3e-15 * perm;
    if ((det > bound || -det > bound) && bound > 1e-290 && bound < 1e290)
        return det > 0 ? 1 : -1;
    const double x[8] = {ax, ay, bx, by, cx, cy, dx, dy};
    // four points on one horizontal or vertical line: every product has a
    // factor that is zero (a difference is zero only for equal numbers)
    if (perm == 0.0 && (ady == 0.0 || bdx == 0.0) && (bdy == 0.0 || adx == 0.0) &&
        (bdy == 0.0 || cdx == 0.0) && (cdy == 0.0 || bdx == 0.0) &&
        (cdy == 0.0 || adx == 0.0) && (ady == 0.0 || cdx == 0.0) && near_exponents<8>(x))
        return 0;
    return incircle_exact(x, bound, err);
}


// ---------------------------------------------------------------------------
// Simulation of Simplicity (Edelsbrunner and Muecke, ACM TOG 9(1), 1990):
// where a predicate is exactly zero, every point i is taken as moved by
// infinitesimals, coordinate c by eps^(2^m(i, c)) with m(i, y) = 3i,
// m(i, x) = 3i + 1 and, for the in-circle lifting z = x^2 + y^2,
// m(i, z) = 3i + 2 (lower indices move more; y before x before z).  The
// perturbed determinant is a polynomial in eps whose terms, largest first,
// have as coefficients +-minors of the unperturbed matrix; the first
// non-zero one gives the sign.  For points sorted by index the order of
// the terms is fixed (the tables below: sign, rows kept, columns kept), so
// no three points are ever collinear and no four cocircular, and
// orientation and in-circle answer for the same perturbed points.
// ---------------------------------------------------------------------------
enum { SOS_ORIENT = 0, SOS_DIFF = 1, SOS_ONE = 2 };
enum { PL_XZ = 0, PL_YZ = 1, PL_XY = 2 };      // planes for SOS_ORIENT
enum { CO_X = 0, CO_Y = 1, CO_Z = 2 };         // coordinates for SOS_DIFF

struct SosTerm {
    signed char sign, kind, r0, r1, r2, what;
};

// orientation of rows (0, 1, 2) of [x y 1] after the determinant itself
static constexpr SosTerm kOrientSos[] = {
    {-1, SOS_DIFF, 1, 2, 0, CO_X},
    {+1, SOS_DIFF, 1, 2, 0, CO_Y},
    {+1, SOS_DIFF, 0, 2, 0, CO_X},
    {+1, SOS_ONE, 0, 0, 0, 0},
};

// in-circle of rows (0, 1, 2, 3) of [x y z 1] after the determinant (terms
// whose minor repeats an earlier one are left out: they are zero when
// reached)
static constexpr SosTerm kIncircleSos[] = {
    {-1, SOS_ORIENT, 1, 2, 3, PL_XZ},
    {+1, SOS_ORIENT, 1, 2, 3, PL_YZ},
    {+1, SOS_ORIENT, 1, 2, 3, PL_XY},
    {+1, SOS_ORIENT, 0, 2, 3, PL_XZ},
    {+1, SOS_DIFF, 2, 3, 0, CO_Z},
    {-1, SOS_DIFF, 2, 3, 0, CO_X},
    {-1, SOS_ORIENT, 0, 2, 3, PL_YZ},
    {+1, SOS_DIFF, 2, 3, 0, CO_Y},
    {-1, SOS_ORIENT, 0, 2, 3, PL_XY},
    {-1, SOS_ORIENT, 0, 1, 3, PL_XZ},
    {-1, SOS_DIFF, 1, 3, 0, CO_Z},
    {+1, SOS_DIFF, 1, 3, 0, CO_X},
    {+1, SOS_DIFF, 0, 3, 0, CO_Z},
    {+1, SOS_ONE, 0, 0, 0, 0},
};

// sorts k indices ascending, permuting the coordinate pairs alongside;
// returns the parity of the permutation (+1 / -1)
template <int K> DT_HD int sort_by_index(int (&idx)[K], double (&x)[2 * K])
{
    int par = 1;
    for (int i = 1; i < K; ++i)
        for (int j = i; j > 0 && idx[j - 1] > idx[j]; --j) {
            const int ti = idx[j]; idx[j] = idx[j - 1]; idx[j - 1] = ti;
            const double tx = x[2 * j], ty = x[2 * j + 1];
            x[2 * j] = x[2 * j - 2]; x[2 * j + 1] = x[2 * j - 1];
            x[2 * j - 2] = tx; x[2 * j - 1] = ty;
            par = -par;
        }
    return par;
}

DT_HD_COLD int orient_sos(const double (&x)[6])
{
    for (const SosTerm &t : kOrientSos) {
        if (t.kind == SOS_ONE) return t.sign;
        const double a = x[2 * t.r0 + t.what], b = x[2 * t.r1 + t.what];
        if (a != b) return a > b ? t.sign : -t.sign;
    }
    return 1;
}

// exact sign of a 2x2 orientation in a plane of (X, Y, Z) among rows r0..r2
DT_HD int lifted_orient(const Big<4> (&U)[4][3], int r0, int r1, int r2, int plane)
{
    const int ca = plane == PL_YZ ? 1 : 0, cb = plane == PL_XY ? 1 : 2;
    const Big<4> a0 = big_sub(U[r0][ca], U[r2][ca]), a1 = big_sub(U[r1][ca], U[r2][ca]);
    const Big<4> b0 = big_sub(U[r0][cb], U[r2][cb]), b1 = big_sub(U[r1][cb], U[r2][cb]);
    return big_sign(big_sub(big_mul<4>(a0, b1), big_mul<4>(b0, a1)));
}

DT_HD_COLD int incircle_sos_wide(const double (&x)[8], int *err)
{
    i128 X[8];
    if (!to_integers<8>(x, X)) {
        set_flag(err, DT_ERR_RANGE);
        return 0;
    }
    // columns x, y, z = x^2 + y^2 at the common scale, as 256-bit integers
    Big<4> U[4][3];
    for (int r = 0; r < 4; ++r) {
        U[r][0] = big_from<4>(X[2 * r]);
        U[r][1] = big_from<4>(X[2 * r + 1]);
        const Big<4> xx = big_mul<2>(big_from<2>(X[2 * r]), big_from<2>(X[2 * r]));
        const Big<4> yy = big_mul<2>(big_from<2>(X[2 * r + 1]), big_from<2>(X[2 * r + 1]));
        U[r][2] = big_add(xx, yy);
    }
    for (const SosTerm &t : kIncircleSos) {
        if (t.kind == SOS_ONE) return t.sign;
        int s;
        if (t.kind == SOS_DIFF)
            s = big_sign(big_sub(U[t.r0][t.what], U[t.r1][t.what]));
        else
            s = lifted_orient(U, t.r0, t.r1, t.r2, t.what);
        if (s) return s * t.sign;
    }
    return 1;
}

// The perturbation's terms as the exact stages above take them: a float64
// evaluation with its bound, then wrapping integers of the size that leaves.
// 2: undecided (the wide evaluation decides).
template <typename U>
DT_HD int lifted_mod(const double (&x)[8], int r0, int r1, int r2, int c, int e)
{
    const int r[3] = {r0, r1, r2};
    U u[3], z[3];
    for (int k = 0; k < 3; ++k) {
        const U X = scaled_mod<U>(x[2 * r[k]], e), Y = scaled_mod<U>(x[2 * r[k] + 1], e);
        u[k] = c ? Y : X;
        z[k] = X * X + Y * Y;
    }
    return sign_mod<U>((u[0] - u[2]) * (z[1] - z[2]) - (z[0] - z[2]) * (u[1] - u[2]));
}

// z of row i less z of row j (z = x^2 + y^2) and the size of its terms
DT_HD double lift_diff(const double (&x)[8], int i, int j, double &size)
{
    const double a = (x[2 * i] - x[2 * j]) * (x[2 * i] + x[2 * j]);
    const double b = (x[2 * i + 1] - x[2 * j + 1]) * (x[2 * i + 1] + x[2 * j + 1]);
    size = __builtin_fabs(a) + __builtin_fabs(b);
    return a + b;
}

// orientation of rows r0, r1, r2 in the plane of (c == 0 ? x : y, z)
DT_HD int lifted_sign(const double (&x)[8], int r0, int r1, int r2, int c, int e)
{
    const double a0 = x[2 * r0 + c] - x[2 * r2 + c], a1 = x[2 * r1 + c] - x[2 * r2 + c];
    if (a0 == 0.0 && a1 == 0.0) return 0;
    double s0, s1;
    const double b0 = lift_diff(x, r0, r2, s0), b1 = lift_diff(x, r1, r2, s1);
    // each lifted difference is off by at most 4.1 u of its size, each
    // product by 6.2 u of the sizes' and the difference by one u more (u =
    // 1.1e-16): 8.1e-16, doubled and rounded up
    const double det = a0 * b1 - b0 * a1;
    const double bound = 2e-15 * (__builtin_fabs(a0) * s1 + __builtin_fabs(a1) * s0);
    if (!(bound > 1e-290 && bound < 1e290)) return 2;
    if (det > bound || -det > bound) return det > 0 ? 1 : -1;
    const int bits = log2_up(bound) + 1 - 3 * e;
    if (bits < 63) return lifted_mod<uint64_t>(x, r0, r1, r2, c, e);
    if (bits < 127) return lifted_mod<u128>(x, r0, r1, r2, c, e);
    return 2;
}

// sign of z of row i less z of row j
DT_HD int lift_diff_sign(const double (&x)[8], int i, int j, int e)
{
    double size;
    const double d = lift_diff(x, i, j, size);
    const double bound = 1e-15 * size;
    if (!(bound > 1e-290 && bound < 1e290)) return 2;
    if (d > bound || -d > bound) return d > 0 ? 1 : -1;
    if (log2_up(bound) + 1 - 2 * e >= 63) return 2;
    const uint64_t X = scaled_mod<uint64_t>(x[2 * i], e), Y = scaled_mod<uint64_t>(x[2 * i + 1], e);
    const uint64_t V = scaled_mod<uint64_t>(x[2 * j], e), W = scaled_mod<uint64_t>(x[2 * j + 1], e);
    return sign_mod<uint64_t>(X * X + Y * Y - V * V - W * W);
}

DT_HD_COLD int incircle_sos(const double (&x)[8], int *err)
{
    int e, span;
    if (!finest_bit<8>(x, e, span) || span > 71) return incircle_sos_wide(x, err);
    for (const SosTerm &t : kIncircleSos) {
        if (t.kind == SOS_ONE) return t.sign;
        int s;
        if (t.kind == SOS_DIFF) {
            if (t.what == CO_Z) {
                s = lift_diff_sign(x, t.r0, t.r1, e);
            } else {
                const double a = x[2 * t.r0 + t.what], b = x[2 * t.r1 + t.what];
                s = a > b ? 1 : a < b ? -1 : 0;
            }
        } else if (t.what == PL_XY) {
            s = orient2d(x[2 * t.r0], x[2 * t.r0 + 1], x[2 * t.r1], x[2 * t.r1 + 1], x[2 * t.r2],
                         x[2 * t.r2 + 1], err);
        } else {
            s = lifted_sign(x, t.r0, t.r1, t.r2, t.what == PL_YZ ? 1 : 0, e);
        }
        if (s == 2) return incircle_sos_wide(x, err);
        if (s) return s * t.sign;
    }
    return 1;
}

// orient2d and incircle of indexed points, never zero for distinct points
// (an exactly degenerate case is decided by the perturbation above)
DT_HD int orient2d_sos(double ax, double ay, double bx, double by, double cx, double cy, int ia,
                       int ib, int ic, int *err)
{
    const int o = orient2d(ax, ay, bx, by, cx, cy, err);
    if (o) return o;
    int idx[3] = {ia, ib, ic};
    double x[6] = {ax, ay, bx, by, cx, cy};
    const int par = sort_by_index<3>(idx, x);
    return par * orient_sos(x);
}

DT_HD int incircle_sos(double ax, double ay, double bx, double by, double cx, double cy,
                       double dx, double dy, int ia, int ib, int ic, int id, int *err)
{
    const int o = incircle(ax, ay, bx, by, cx, cy, dx, dy, err);
    if (o) return o;
    int idx[4] = {ia, ib, ic, id};
    double x[8] = {ax, ay, bx, by, cx, cy, dx, dy};
    const int par = sort_by_index<4>(idx, x);
    return par * incircle_sos(x, err);
}

}  // namespace dt
}  // namespace cvt
