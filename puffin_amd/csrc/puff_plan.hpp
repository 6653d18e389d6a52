// Plain C++ of the library, shared by kernels and host code and compiled alone
// by the tests: index arithmetic of the mesh, bounds, the propagator's sine and
// cosine, plans of the FFT lines.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define PUFF_BOTH __host__ __device__ __forceinline__
#else
#define PUFF_BOTH inline
#endif

namespace puff {

// Component (0: real, 1: imaginary) of a node in an interleaved mesh, counted
// in components.  Meshes hold up to 2^31 - 1 nodes: twice that is past an int.
PUFF_BOTH uint32_t node_component(int node, int part) { return 2u * (uint32_t)node + (uint32_t)part; }

// Largest (kx^2 + ky^2) / |2 kz| over the wavenumbers with kz != 0 (0 if none).
template <typename V>
double largest_phase_rate(const V& kx, const V& ky, const V& kz) {
    auto largest = [](const V& k) {
        double m = 0.0;
        for (double v : k) m = std::max(m, v * v);
        return m;
    };
    const double k2 = largest(kx) + largest(ky);
    double rate = 0.0;
    for (double v : kz)
        if (v != 0.0) rate = std::max(rate, k2 * std::fabs(1.0 / (2.0 * v)));
    return rate;
}

// Sine and cosine of the propagator's phase, an FP64 number below PHASE_LIMIT:
// reduced by multiples n of pi / 2 (a double and its remainder, each product
// in one FMA: exact to 1e-17 while n is), then Taylor sums.  FP64: to x^17 and
// x^18, with the rounding errors of the reduction and of x^2 carried along:
// within 9.5e-17 of the true values up to 3e13 (half an ulp of 1 is 1.1e-16).
// FP32: the rotated field is rounded to 6e-8 anyway; sums to x^9 and x^10 of the
// reduced phase rounded to FP32 (|r| <= pi / 4): within 7.5e-8.  40 and 20
// instructions without branches; the library's functions carry a second path for
// large arguments at each of their places in a kernel.
constexpr double PHASE_LIMIT = 1e13;   // n stays below 2^43
template <typename R>
struct SinCos {
    R s, c;
};
template <typename R>
PUFF_BOTH SinCos<R> sincos_phase(double th) {
    constexpr double hi = 1.57079632679489661923, lo = 6.123233995736766036e-17;
    const double n = rint(th * 0.63661977236758134308);
    const double r0 = fma(-n, hi, th);
    const double r = fma(-n, lo, r0);
    R sn, cs;
    if constexpr (sizeof(R) == 8) {
        const double e = fma(-n, lo, r0 - r);
        const double z = r * r;
        double p = fma(z, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
        p = fma(z, p, 1.0 / 6227020800.0);
        p = fma(z, p, -1.0 / 39916800.0);
        p = fma(z, p, 1.0 / 362880.0);
        p = fma(z, p, -1.0 / 5040.0);
        p = fma(z, p, 1.0 / 120.0);
        p = fma(z, p, -1.0 / 6.0);
        sn = r + fma(r * z, p, e);
        double q = fma(z, -1.0 / 6402373705728000.0, 1.0 / 20922789888000.0);
        q = fma(z, q, -1.0 / 87178291200.0);
        q = fma(z, q, 1.0 / 479001600.0);
        q = fma(z, q, -1.0 / 3628800.0);
        q = fma(z, q, 1.0 / 40320.0);
        q = fma(z, q, -1.0 / 720.0);
        q = fma(z, q, 1.0 / 24.0);
        const double hz = 0.5 * z, w = 1.0 - hz;
        cs = w + fma(z * z, q, fma(-r, e, fma(-0.5, fma(r, r, -z), (1.0 - w) - hz)));
    } else {
        const float x = (float)r, z = x * x;
        float p = fmaf(z, 1.0f / 362880.0f, -1.0f / 5040.0f);
        p = fmaf(z, p, 1.0f / 120.0f);
        p = fmaf(z, p, -1.0f / 6.0f);
        sn = fmaf(x * z, p, x);
        float q = fmaf(z, -1.0f / 3628800.0f, 1.0f / 40320.0f);
        q = fmaf(z, q, -1.0f / 720.0f);
        q = fmaf(z, q, 1.0f / 24.0f);
        q = fmaf(z, q, -0.5f);
        cs = fmaf(z, q, 1.0f);
    }
    const int m = (int)(int64_t)n;
    const R a = (m & 1) ? cs : sn, b = (m & 1) ? sn : cs;
    return {(m & 2) ? -a : a, ((m + 1) & 2) ? -b : b};
}

// ---- FFT lines ----------------------------------------------------------------

inline bool is_prime(int n) {
    if (n < 2) return false;
    for (int f = 2; (int64_t)f * f <= n; ++f)
        if (n % f == 0) return false;
    return true;
}

// Lines by Rader's algorithm: n prime and n - 1 a power of two, 257 among the
// admitted lengths.  17 points run faster and closer to the exact transform as
// one pass of direct sums on the matrix cores: a diffraction step of
// 17 x 17 x 200 takes 84 us against 138 (FP64; errors 3.7e-16 and 4.3e-16
// r.m.s.), of 17 x 17 x 4096 (mixed) 255 against 447 us.
inline bool rader_line(int n) { return n > 17 && is_prime(n) && ((n - 1) & (n - 2)) == 0; }

// Fewest radices of 2 to 16, each at most `top` and in falling order, with
// product m (the smallest largest one where the count is the same); the number
// of them, or 99.
inline int radices(int m, int top, int* out) {
    if (m == 1) return 0;
    int best = 99;
    for (int r = 2; r <= top && r <= m; ++r) {
        if (m % r) continue;
        int rest[32];
        const int k = 1 + radices(m / r, r, rest);
        if (k < best) {
            best = k;
            out[0] = r;
            std::copy(rest, rest + k - 1, out + 1);
        }
    }
    return best;
}

// Passes of an n-point transform: prime factors above 13 as direct passes, the
// rest in the fewest passes of up to 16 points (every pass is a round trip
// through LDS and a barrier): 420 = 10 x 7 x 6, 90 = 10 x 9, 75 = 15 x 5.
template <typename Axis>
void factorize(int n, Axis& ax) {
    ax.n = n;
    ax.npass = 0;
    int m = n;
    for (int f : {2, 3, 5, 7, 11, 13})
        while (m % f == 0) m /= f;
    const int small = n / m;
    int big[32];
    int nbig = 0;
    for (int f = 17; m > 1 && (int64_t)f * f <= m; f += 2)
        while (m % f == 0) { big[nbig++] = f; m /= f; }
    if (m > 1) big[nbig++] = m;
    for (int k = nbig - 1; k >= 0; --k) ax.radix[ax.npass++] = big[k];
    int r[32];
    const int k = radices(small, 16, r);
    for (int q = 0; q < k; ++q) ax.radix[ax.npass++] = r[q];
}

// LDS word of flat element e of a line-major buffer (IL false): one spare
// slot after every 16 elements.  A radix-16 pass with p = 1 has each lane
// write 16 consecutive outputs, so lanes write 16 elements apart, all on the
// same LDS banks; with the spare slots they land 17 apart and 16 lanes cover
// all the banks.  Interleaved buffers (IL: y and z2 lines, b fastest) put
// consecutive lanes on consecutive elements and are not padded.
#ifndef PUFF_LDS_PAD_X
#define PUFF_LDS_PAD_X 1
#endif
template <bool IL>
PUFF_BOTH constexpr int lpad(int e) {
    return (!IL && PUFF_LDS_PAD_X) ? e + (e >> 4) : e;
}

// How a runtime plan runs (line_plan): all passes of at most 16 points, in
// place; a large prime first, on the matrix cores, then the same; or with two
// line buffers.  A kernel each: the matrix pass's accumulators take a
// wavefront per SIMD from the others.
enum { LINE_SMALL = 0, LINE_PRIME = 1, LINE_TWO = 2 };

constexpr int MFMA_TILES = 4;
constexpr int mfma_tiles(int B, int n, int r) { return (B * (n / r) + 7) / 8 * (((r - 1) / 2 + 16) / 16); }

// Lines per workgroup (B) and the plan's kind.  In place every pass's
// butterflies must fit the threads' registers (radix_pass) and the matrix
// pass's tiles their accumulators; where one line already does not, or a plan
// has Rader's or a second large prime, two buffers.  tw: the twiddle table in
// LDS too (x and y lines).  Both sides of the line, one diffraction step:
// 90 x 75 x 420 (FP64) 816 us in two buffers with direct sums of 5 and 7,
// 364 us in place; 61 x 47 x 389 640 us with direct sums, 375 us on the matrix
// cores; 76 x 42 x 457 (mixed) 615 and 335 us.  The matrix pass forms tiles of 8
// butterflies however few a workgroup has: with 3 of them (61 x 57 x 1047, FP64)
// 820 us against 1430 in two buffers, with 2 (100 x 90 x 958) 3880 against 3350.
#ifndef PUFF_Z_LDS_BUDGET
#define PUFF_Z_LDS_BUDGET (32 * 1024)
#endif
#ifndef PUFF_XY_LDS_BUDGET
#define PUFF_XY_LDS_BUDGET (32 * 1024)
#endif
#ifndef PUFF_Y_LDS_BUDGET
#define PUFF_Y_LDS_BUDGET PUFF_XY_LDS_BUDGET
#endif
constexpr int lines_per_block(int n, size_t elem, int cap, size_t budget, bool il, bool two, int table) {
    int b = cap;
    while (b > 1 && ((two ? 2 : 1) * (size_t)(il ? lpad<true>(b * n) : lpad<false>(b * n)) + table) * elem > budget)
        --b;
    return b;
}
constexpr int PRIME_LEAST = 3;
struct LinePlan {
    int B, kind;
};

// Half the lines a workgroup, and half again, down to `least`, while the mesh's
// rows of `cols` lines give work to fewer than three quarters of the CUs.  A
// diffraction step of 26 x 26 x 236 (FP64; 52 workgroups of 15 z2 lines else)
// 146 -> 107 us; with two workgroups a CU as the aim, small lines lose
// (26 x 26 x 260: 116 -> 121 us).
constexpr int CUS = 256;
inline int filled(int B, int least, int64_t cols, int64_t rows) {
    while (B / 2 >= least && (cols + B - 1) / B * rows < 3 * CUS / 4) B /= 2;
    return B;
}

template <typename Axis>
LinePlan line_plan(const Axis& ax, size_t elem, int cap, size_t budget, bool il, bool tw, int64_t cols, int64_t rows) {
    int kind = ax.rader ? LINE_TWO : LINE_SMALL;
    int fit = cap;   // lines whose butterflies fit the registers
    for (int k = 0; k < ax.npass; ++k) {
        const int r = ax.radix[k];
        if (r > 16 && k > 0) {
            kind = LINE_TWO;
        } else if (r > 16) {
            if (kind == LINE_SMALL) kind = LINE_PRIME;
            while (fit > 0 && mfma_tiles(fit, ax.n, r) > 4 * MFMA_TILES) --fit;
        } else {
            fit = std::min(fit, (16 / r) * 256 / (ax.n / r));
        }
    }
    if (fit < 1) kind = LINE_TWO;
    const int table = tw ? ax.n : 0;
    if (kind == LINE_PRIME) {
        // whole tiles of 8 butterflies, where 64 KiB have room for them
        const int r = ax.radix[0], T = ax.n / r, whole = (8 + T - 1) / T;
        auto lines = [&](int most, size_t room) { return lines_per_block(ax.n, elem, most, room, il, false, table + r); };
        int B = lines(fit, lines(whole, 2 * budget) == whole ? 2 * budget : budget);
        if (8 % T == 0 && B > whole) B -= B % whole;   // no part-filled tile
        if (B * T >= PRIME_LEAST) return {filled(B, std::min(B, whole), cols, rows), kind};
        kind = LINE_TWO;
    }
    if (kind == LINE_TWO) return {lines_per_block(ax.n, elem, cap, budget, il, true, table), kind};
    return {filled(lines_per_block(ax.n, elem, fit, budget, il, false, table), 1, cols, rows), kind};
}

constexpr size_t LDS_BYTES = 160 * 1024;   // of a CU, all of it one workgroup's at most

// LDS bytes of a workgroup of B lines of an axis (0: x, 1: y, 2: z2).
template <typename Axis>
size_t line_lds(const Axis& ax, int B, int kind, size_t elem, int axis) {
    const size_t line = axis ? lpad<true>(B * ax.n) : lpad<false>(B * ax.n);
    const int table = (axis < 2 ? ax.n : 0) + (kind == LINE_PRIME ? ax.radix[0] : 0);
    return ((kind == LINE_TWO ? 2 : 1) * line + table) * elem;
}

// The runtime plan of an axis.
template <typename Axis>
LinePlan axis_plan(const Axis& ax, size_t elem, int axis, int64_t cols, int64_t rows) {
    if (axis == 0) return line_plan(ax, elem, 64, PUFF_XY_LDS_BUDGET, false, true, cols, rows);
    if (axis == 1) return line_plan(ax, elem, 16, PUFF_Y_LDS_BUDGET, true, true, cols, rows);
    return line_plan(ax, elem, 16, PUFF_Z_LDS_BUDGET, true, false, cols, rows);
}

// Whether a workgroup holds one line of the axis's plan.  A context admits
// lines of three times n elements (two buffers and the table); the spare slots
// of x lines in two buffers take another n / 8.
template <typename Axis>
bool line_fits(const Axis& ax, size_t elem, int axis) {
    const LinePlan lp = axis_plan(ax, elem, axis, 1, 1);
    return line_lds(ax, lp.B, lp.kind, elem, axis) <= LDS_BYTES;
}

}  // namespace puff
