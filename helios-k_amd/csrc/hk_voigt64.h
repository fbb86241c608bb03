// hk_voigt64.h -- the plain FP64 form of the Voigt sum: one workgroup sums
// the lines of one tile of the grid (owner computes, no atomics).
//
// The sum over a tile is split by how smooth a line is over it, not by how
// far the lines' windows reach:
//   * tile level: a line whose cut window covers the tile and whose centre
//     lies >= kFarRatio64 tile half widths from the tile's centre (with
//     x^2 + y^2 >= 100 over the tile) is analytic over it; it is evaluated
//     at the tile's 20 Chebyshev-Gauss nodes only, one line per lane, the
//     node sums kept in that lane's registers;
//   * wave level: the same over the 64 PPT points of one wave, for the lines
//     the tile level leaves (nearer centres, windows that end in the tile);
//   * the rest is evaluated point by point, one line per wave at a time, 64
//     points per instruction.
// The node sums become one Chebyshev series per wave (the tile's series is
// carried to the wave's nodes), evaluated once per point in FP64.
//
// Truncation: the worst line (centre at the band's inner edge, zero width:
// a double pole) interpolates to 3.3e-16 of its value, largest at the tile end
// nearest the line; everything else is FP64 rounding, as in the pair sum (one
// line alone: 1.3e-15 of its value at most, pair by pair 9e-16; sums of 20000
// lines 2e-15, pair by pair 1e-14).  At 3.25 half widths 5e-15 were left, for
// 1 to 5 % less time.
// The nodes and the points are placed relative to the tile centre, so the
// rounding of x_j = fma(j, dnu, numin) enters the far field exactly as it
// enters a pair.
//
// What bounds it: FP64 vector instructions.  At 1e5 lines, 3e6 points, cut
// 100 cm^-1 a line has 2e4 pairs in its window; it takes 20 node values in
// each of ~17 tiles, 20 in ~9 waves and ~13 segments of 64 points -- 30 times
// fewer evaluations than pairs.  Pair by pair (with a separate line-core
// pass) that spectrum took 2217 us, now 497; 2.35e6 lines on 7e6 points at
// 10 bar, cut 25: 132 ms, now 15.8.
#pragma once
#include <type_traits>

#include "hk_device.h"
#include "hk_tiles.h"

namespace hk {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

constexpr int kFN64 = 20;                 // Chebyshev-Gauss nodes
constexpr double kFarRatio64 = 3.7;
// Largest x^2 + y^2 of a far line: keeps the products of the 8-node rule
// (~ r2^16 for a pair of nodes) in range.
constexpr double kFarMaxR2 = 1.0e18;
// cos(j pi / 40), j = 0..20, correctly rounded: a table of cospi(j / 40.0), whose
// argument rounds, put 3e-15 of a far line on the tile's ends
__device__ constexpr double kCos40[kFN64 + 1] = {
    1.0, 0.996917333733128, 0.9876883405951378, 0.9723699203976766, 0.9510565162951535,
    0.9238795325112867, 0.8910065241883679, 0.8526401643540922, 0.8090169943749475,
    0.7604059656000309, 0.7071067811865476, 0.6494480483301837, 0.5877852522924731,
    0.5224985647159489, 0.4539904997395468, 0.3826834323650898, 0.30901699437494745,
    0.23344536385590542, 0.15643446504023087, 0.07845909572784494, 0.0};
// cos(j pi / 40), 0 <= j < 80
__device__ __forceinline__ double cos40(int j) {
    const int q = j > 2 * kFN64 ? 4 * kFN64 - j : j;
    return q > kFN64 ? -kCos40[2 * kFN64 - q] : kCos40[q];
}
// Chebyshev-Gauss node k of 20, cos(pi (k + 1/2) / 20)
__device__ __forceinline__ double node_u(int k) { return cos40(2 * k + 1); }
// Points per thread of a tile (256 threads) when the caller leaves it open.
// Halving the tile doubles the tile-level node evaluations and halves the point
// sums; 512 points win over 1024 at 1e5 lines, 3e6 points, cut 100 (492 against
// 542 us), 5e6 lines (16.4 / 20.4 ms), 3.3e5 lines, 1e6 points (1.06 / 1.40 ms) and
// 2.35e6 lines, 7e6 points, cut 25 on a 0.001 cm^-1 grid (15.9 / 16.4 ms).
// Grids of fewer than four 512-point tiles per CU take 256-point tiles: 1e4
// points 67 against 110 us, 1e5 lines of cut 100 on 3e4 points 1.13 / 2.34 ms, on
// 3e5 points 430 / 468 us; at 1e6 points the two are equal.
// With every pair evaluated, longer grids take 1024 or 2048 points, so that a
// line's broadcast serves four or eight points a lane (tiles of 512, 1024 and 2048
// points: 24 spectra of 3e6 points, 1e4 to 5e6 lines, 684, 559 and 535 ms; 1e5
// lines, 3e6 points 2.12, 2.01 and 1.92 ms; 2.35e6 lines at 10 bar, 7e6 points 128,
// 115 and 126 ms).  Below 1024 tiles of 2048 points the chip is not full.
inline int64_t tiles64(int64_t nx, int ppt) { return (nx + kThreads * ppt - 1) / (kThreads * ppt); }
// Sparse lists, at most two lines per 512 points on average, have kernels of their
// own that take a tile of few lines point by point: its nodes, of which a line or
// two fill one lane each, their series and the registers spilled around them took
// most of the time (500 lines, 3e6 points, cut 25: 78 us, 34 without; 5000 lines
// 147 and 90).  In the kernel for all lists the second path costs dense ones 2 to
// 9 %.
inline bool sparse64(int64_t nx, int64_t nl) {
    return nl <= 2 * tiles64(nx, 2) && tiles64(nx, 2) >= 512;
}
inline int default_ppt64(int64_t nx, int64_t nl, bool exact) {
    if (!exact && sparse64(nx, nl)) return 2;
    if (tiles64(nx, 2) < 1024) return 1;
    return !exact ? 2 : tiles64(nx, 8) < 1024 ? 4 : 8;
}
// The width a caller asks for is kept where it can be of use: 4096 points are
// taken as 2048 (16 sums a lane leave two waves a SIMD: 1e5 lines, 3e6 points 1.97
// and 0.81 ms, every pair 3.31 and 1.92), more than 1024 need a tile for each CU
// (1e4 points, 2000 lines, every pair: 1024 points 428 us, 2048 1086), and with
// every pair evaluated 512 are taken as 1024 where those fill the chip (above).
inline int asked_ppt64(int ppt, int64_t nx, bool exact) {
    if (exact && ppt == 2 && tiles64(nx, 4) >= 1024) return 4;
    if (ppt > 8) ppt = 8;
    return ppt == 8 && tiles64(nx, 8) < 256 ? 4 : ppt;
}

// Tiles of a sparse list that at most this many lines can reach.
constexpr int kFewLines = 32;

// lines taken per round of the tile loop (each wave lists its own quarter)
constexpr int kRound64 = 4096;
// a chunk of 64 lines goes through the wave's nodes when at least this many
// of them qualify (20 node evaluations against PPT per line)
constexpr int wave_min_lines(int ppt) { return kFN64 / ppt + 2; }

struct Far64LDS {
    uint16_t list[kWaves][kRound64 / kWaves];   // near lines, relative to the round
    double F[kWaves][kFN64];                    // tile node sums, one row per wave
    double wF[kWaves][kFN64];                   // wave node sums, then its series
    double c[kWaves][kFN64];                    // tile series (a copy per wave)
    double tab[kWaves][64];                     // core table of the wave's line
    double cosv[4 * kFN64];                     // cos(j pi / 40)
    uint64_t taken[kWaves][kRound64 / 64];      // lines of a chunk the wave's nodes took
    double cst[kWaves];                         // plinths alone: of lines that cover the tile
    int cnt[kWaves];
    int64_t range[2];
};

// Orders a wave's own LDS writes before its later reads of them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A uniform constant the compiler cannot hoist: the unrolled node loops use
// dozens of FP64 literals, and kept in scalar registers across the tile loop
// they spill.
__device__ __forceinline__ double local_const(double v) {
    asm volatile("" : "+s"(v));
    return v;
}

// e^v for |v| <= 0.35 by its Taylor series (first term left out < 3e-18).
__device__ __forceinline__ double exp_small(double v) {
    constexpr double c[14] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040,
                              1.0 / 40320, 1.0 / 362880, 1.0 / 3628800, 1.0 / 39916800,
                              1.0 / 479001600, 1.0 / 6227020800};
    double s = local_const(c[13]);
#pragma unroll
    for (int k = 12; k >= 2; --k) s = fma(s, v, local_const(c[k]));
    return fma(fma(s, v, 1.0), v, 1.0);
}

// e^-t, |t| <= 800 (t = n ln 2 - v in two parts).
__device__ __forceinline__ double exp_neg(double t) {
    const double n = rint(t * local_const(1.4426950408889634));
    double v = fma(n, local_const(0.69314718055994531), -t);
    v = fma(n, local_const(2.3190468138462996e-17), v);
    return ldexp(exp_small(v), -(int)n);
}

__device__ __forceinline__ double swap_add32(double a, double b) {
    // lanes < 32: a summed over (lane, lane + 32); lanes >= 32: b likewise
    const uint64_t x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false,
                                                    false);
    return __longlong_as_double(((uint64_t)h[0] << 32) | l[0]) +
           __longlong_as_double(((uint64_t)h[1] << 32) | l[1]);
}

__device__ __forceinline__ double swap_add16(double a, double b) {
    // even rows of 16 lanes: a summed over the row and the next; odd rows: b
    const uint64_t x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false,
                                                    false);
    return __longlong_as_double(((uint64_t)h[0] << 32) | l[0]) +
           __longlong_as_double(((uint64_t)h[1] << 32) | l[1]);
}

template <int CTRL>
__device__ __forceinline__ double row_dpp64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Wave totals of the 20 per-lane sums f, added to row[].  Halving exchanges
// (two values share one register after each) take 105 instructions where 20
// separate wave sums take 360.  Fixed order: deterministic.  All lanes active.
__device__ __forceinline__ void add_node_totals(const double (&f)[kFN64], double *row) {
    const int lane = threadIdx.x & 63;
    double z[kFN64 / 4];
#pragma unroll
    for (int q = 0; q < kFN64 / 4; ++q)
        z[q] = swap_add16(swap_add32(f[4 * q], f[4 * q + 1]), swap_add32(f[4 * q + 2], f[4 * q + 3]));
    double mine = 0.0;
    const int p = lane & 15;
#pragma unroll
    for (int q = 0; q < kFN64 / 4; ++q) {
        double v = z[q];
        v += row_dpp64<0xb1>(v);     // quad_perm [1,0,3,2]
        v += row_dpp64<0x4e>(v);     // quad_perm [2,3,0,1]
        v += row_dpp64<0x141>(v);    // row_half_mirror
        v += row_dpp64<0x140>(v);    // row_mirror
        mine = p == q ? v : mine;
    }
    // rows 0, 1, 2, 3 of 16 lanes hold nodes 4q, 4q + 2, 4q + 1, 4q + 3
    const int r = lane >> 4;
    if (p < kFN64 / 4) row[4 * p + (r == 1 ? 2 : r == 2 ? 1 : r)] += mine;
}

// Sub-Lorentzian factor of the wings (hk_chi): for lo < x < hi a line's value is
// multiplied by chi(|x - nu|) x / nu.
struct Chi {
    double s1, s2, s3, B1, B2, B3, lo, hi;
};

// -ln chi at distance d (Perrin & Hartmann 1989).
__device__ __forceinline__ double chi_exponent(const Chi &c, double d) {
    if (d < c.s1) return 0.0;
    if (d < c.s2) return c.B1 * (d - c.s1);
    if (d < c.s3) return fma(c.B1, c.s2 - c.s1, c.B2 * (d - c.s2));
    return fma(c.B1, c.s2 - c.s1, fma(c.B2, c.s3 - c.s2, c.B3 * (d - c.s3)));
}

// The factor over an interval on which it is one analytic piece, at u of its
// half widths from its centre: exp(-(B (x - nu) + t0)) (c + u h), c + u h = x / nu
// (1 + (x - nu) / nu would cancel far below the line); 1 outside the range.
struct ChiPiece {
    double B = 0.0, t0 = 0.0, c = 1.0, h = 0.0;
};

// Finds the piece for the points xa..xb (D: the interval's centre from the
// line's); false when they straddle a break or an end of the range, or when the
// exponential varies too much for the nodes (|B| half <= 2 leaves 1e-18).
__device__ __forceinline__ bool chi_piece(const Chi &c, double xa, double xb, double nu, double D,
                                          double half, ChiPiece &p) {
    p = ChiPiece();
    if (xb <= c.lo || xa >= c.hi) return true;
    if (!(xa > c.lo && xb < c.hi)) return false;
    const double d0 = fabs(D) - half, d1 = fabs(D) + half;
    double B, t0;
    if (d1 <= c.s1) { B = 0.0; t0 = 0.0; }
    else if (d0 >= c.s1 && d1 <= c.s2) { B = c.B1; t0 = -c.B1 * c.s1; }
    else if (d0 >= c.s2 && d1 <= c.s3) { B = c.B2; t0 = fma(c.B1, c.s2 - c.s1, -c.B2 * c.s2); }
    else if (d0 >= c.s3) {
        B = c.B3;
        t0 = fma(c.B1, c.s2 - c.s1, fma(c.B2, c.s3 - c.s2, -c.B3 * c.s3));
    } else return false;
    p.B = D < 0.0 ? -B : B;
    p.t0 = t0;
    const double inv_nu = 1.0 / nu;
    p.c = 0.5 * (xa + xb) * inv_nu;
    p.h = half * inv_nu;
    return fabs(B) * half <= 2.0;
}

// What a line contributes to a point: PROFILE 1 Voigt, 2 Lorentz, 3 Doppler,
// 4 binned Gaussian, 0 nothing but the plinth; PLINTH subtracts the line's
// value at its cut (args.pl) over its whole window; CHI applies args.chi.
// WHOLE: lines that have one wing formula over all of a wave's points take
// add_wing.  EXACT: every pair is evaluated, nothing goes through nodes.
// SPARSE: tiles of few lines take them point by point, each wave by itself.
template <int PROFILE_, bool PLINTH_, bool CHI_, bool WHOLE_ = false, bool EXACT_ = false,
          bool SPARSE_ = false>
struct LineSum {
    static constexpr int PROFILE = PROFILE_;
    static constexpr bool PLINTH = PLINTH_, CHI = CHI_, WHOLE = WHOLE_, EXACT = EXACT_;
    static constexpr bool SPARSE = SPARSE_;
    // wings that the nodes can take, or a value that underflows to zero beyond
    // x = kDopplerEnd (e^-x^2 does at 27.3)
    static constexpr bool WINGS = PROFILE == 1 || PROFILE == 2;
    static constexpr bool COMPACT = PROFILE == 3 || PROFILE == 4;
};
constexpr double kDopplerEnd = 27.5;

// The factor G of a line's profile value.
template <class P>
__device__ __forceinline__ double line_factor(double S, double y) {
    if (P::PROFILE == 1) return S * kISqrtPi * y * (2.0 / kPi);
    if (P::PROFILE == 2) return S * y / kPi;
    return P::PROFILE == 3 ? S * kISqrtPi : P::PROFILE == 4 ? S : 0.0;
}

__device__ __forceinline__ double lane_f64(double v, int b) {
    const long long x = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)x, b);
    const unsigned hi = __builtin_amdgcn_readlane((int)(x >> 32), b);
    return __longlong_as_double(((long long)hi << 32) | lo);
}

// Sum of v over the wave (fixed order), in every lane.
__device__ __forceinline__ double wave_total64(double v) {
    v += row_dpp64<0xb1>(v);
    v += row_dpp64<0x4e>(v);
    v += row_dpp64<0x141>(v);
    v += row_dpp64<0x140>(v);
    return ((lane_f64(v, 0) + lane_f64(v, 16)) + lane_f64(v, 32)) + lane_f64(v, 48);
}

// Far class of a line for an interval of half width `half` whose centre lies
// D from the line centre [cm^-1]: 0 = not far, else the wing formula its
// nearest point allows (1 series, 2 four nodes, 3 eight nodes; Lorentz has one
// formula).
template <class P>
__device__ __forceinline__ int far_class64(double D, double half, double ia, double y2, double G) {
    if (!P::WINGS) return 0;
    const double d = fabs(D);
    const double xn = (d - half) * ia, xf = (d + half) * ia;
    const double rn = fma(xn, xn, y2), rf = fma(xf, xf, y2);
    const bool ok = d >= kFarRatio64 * half && fabs(G) < 1.0e300;
    if (P::PROFILE == 2) return ok && rn > 0.0 && rf < 1.0e150 ? 1 : 0;
    return !(ok && rn >= kRB64 && rf < kFarMaxR2) ? 0 : rn >= kRF64 ? 1 : rn >= kRM64 ? 2 : 3;
}

// Constants of the two Gauss-Hermite rules (gh4_sum64, gh8_sum64): squared
// nodes, -4 times them, weights.
template <int N>
struct GH {
    double a[N], m4a[N], w[N];
    __device__ __forceinline__ GH() {
        constexpr double t4[2] = {kGH4t1, kGH4t2}, w4[2] = {kGH4w1, kGH4w2};
        constexpr double t8[4] = {kGH8t1, kGH8t2, kGH8t3, kGH8t4};
        constexpr double w8[4] = {kGH8w1, kGH8w2, kGH8w3, kGH8w4};
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const double t = N == 2 ? t4[k & 1] : t8[k];
            a[k] = local_const(t * t);
            m4a[k] = local_const(-4.0 * t * t);
            w[k] = local_const(N == 2 ? w4[k & 1] : w8[k]);
        }
    }
};

// Numerator and denominator of sum_k w_k u_k / D_k.
__device__ __forceinline__ void gh_frac(const GH<2> &q, double x2, double r2, double &num,
                                        double &den) {
    const double u1 = r2 + q.a[0], u2 = r2 + q.a[1];
    const double D1 = fma(u1, u1, q.m4a[0] * x2);
    const double D2 = fma(u2, u2, q.m4a[1] * x2);
    num = fma(q.w[0] * u1, D2, q.w[1] * u2 * D1);
    den = D1 * D2;
}

__device__ __forceinline__ void gh_frac(const GH<4> &q, double x2, double r2, double &num,
                                        double &den) {
    const double u1 = r2 + q.a[0], u2 = r2 + q.a[1], u3 = r2 + q.a[2], u4 = r2 + q.a[3];
    const double D1 = fma(u1, u1, q.m4a[0] * x2);
    const double D2 = fma(u2, u2, q.m4a[1] * x2);
    const double D3 = fma(u3, u3, q.m4a[2] * x2);
    const double D4 = fma(u4, u4, q.m4a[3] * x2);
    const double D12 = D1 * D2, D34 = D3 * D4;
    const double n12 = fma(q.w[0] * u1, D2, q.w[1] * u2 * D1);
    const double n34 = fma(q.w[2] * u3, D4, q.w[3] * u4 * D3);
    num = fma(n12, D34, n34 * D12);
    den = D12 * D34;
}

// One line's values at the 20 nodes of an interval (centre D from the line
// centre, half width half), added to f.  The nodes +-u_k share one
// reciprocal.  g: line_factor, pl: the plinth (0 for a lane without a line),
// taken off here, before any sum, as from a pair.
template <class P, int CLASS>
__device__ __forceinline__ void add_nodes(double D, double half, double ia, double y2, double g,
                                          double pl, const ChiPiece &chi, double (&f)[kFN64]) {
    const double xc = D * ia, h = half * ia;
    double p2 = 0.0, p3 = 0.0, p4 = 0.0;
    if (P::PROFILE == 1 && CLASS == 1) {
        p2 = fma(-2.0, y2, 3.75); p3 = -15.0 * y2; p4 = 12.0 * y2 * y2;
        g *= 0.5 * kPi * kISqrtPi;      // S y / pi
    }
    const GH<CLASS == 3 ? 4 : 2> gh;
#pragma unroll
    for (int k = 0; k < kFN64 / 2; ++k) {
        __builtin_amdgcn_sched_barrier(0);   // (pairs interleaved: spills)
        const double u = local_const(kCos40[2 * k + 1]);
        const double xa = fma(u, h, xc), xb = fma(-u, h, xc);
        const double a2 = xa * xa, b2 = xb * xb;
        const double ra = a2 + y2, rb = b2 + y2;
        double va, vb;
        if (P::PROFILE == 2) {
            const double q = rcp64(ra * rb);
            va = q * rb;
            vb = q * ra;
        } else if (CLASS == 1) {
            const double q = rcp64(ra * rb), ia1 = q * rb, ib1 = q * ra;
            va = ia1 * fma(fma(fma(fma(p4, ia1, p3), ia1, p2), ia1, 1.5), ia1, 1.0);
            vb = ib1 * fma(fma(fma(fma(p4, ib1, p3), ib1, p2), ib1, 1.5), ib1, 1.0);
        } else {
            double na, da, nb, db;
            gh_frac(gh, a2, ra, na, da);
            gh_frac(gh, b2, rb, nb, db);
            const double q = rcp64(da * db);
            va = na * db * q;
            vb = nb * da * q;
        }
        if (P::CHI) {
            const double ea = fma(u, half, D), eb = fma(-u, half, D);
            va *= exp_neg(fma(chi.B, ea, chi.t0)) * fma(u, chi.h, chi.c);
            vb *= exp_neg(fma(chi.B, eb, chi.t0)) * fma(-u, chi.h, chi.c);
        }
        // (g last: strengths far below 1e-100 must not meet the products)
        if constexpr (P::PLINTH) {
            f[k] += fma(g, va, -pl);
            f[kFN64 - 1 - k] += fma(g, vb, -pl);
        } else {
            f[k] = fma(g, va, f[k]);
            f[kFN64 - 1 - k] = fma(g, vb, f[kFN64 - 1 - k]);
        }
    }
}

// The lanes with cls != 0 add their lines' node values; the whole wave takes
// the formula of the line nearest its interval (valid farther out too).
template <class P>
__device__ __forceinline__ void add_far_lines(int cls, double D, double half, double ia, double y2,
                                              double G, double pl, const ChiPiece &chi,
                                              double (&f)[kFN64]) {
    if (!P::WINGS || __ballot(cls != 0) == 0ull) return;
    if (cls == 0) { D = 1.0; half = 0.0; ia = 1.0e4; y2 = 0.0; G = 0.0; pl = 0.0; }
    if (P::PROFILE == 1 && __ballot(cls == 3)) add_nodes<P, 3>(D, half, ia, y2, G, pl, chi, f);
    else if (P::PROFILE == 1 && __ballot(cls == 2)) add_nodes<P, 2>(D, half, ia, y2, G, pl, chi, f);
    else add_nodes<P, 1>(D, half, ia, y2, G, pl, chi, f);
}

// First index p of [0, n) with !(v[p] < key) (LOWER) or v[p] > key, by one
// wave: 64 probes per step, so 1e7 keys take four dependent loads.
template <bool LOWER>
__device__ __forceinline__ int64_t wave_bound(const double *__restrict__ v, int64_t n, double key) {
    const int lane = threadIdx.x & 63;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t step = (hi - lo + 63) >> 6;
        const int64_t p = lo + lane * step;
        bool below = false;
        if (p < hi) { const double x = v[p]; below = LOWER ? x < key : x <= key; }
        const int c = __popcll(__ballot(below));
        if (c == 0) break;
        hi = min(hi, lo + c * step);
        lo += (c - 1) * step + 1;
    }
    return lo;
}

// Window [lo, hi) of a line on the n points from jb on: |x_j - nu| < hw in
// FP64, the set cut_window finds (the estimate is stepped until both
// predicates flip).
__device__ __forceinline__ void clip_window(double nu, double hw, double numin, double dnu,
                                            double inv_dnu, int64_t jb, int n, int &lo, int &hi) {
    if (!(hw > 0.0)) { lo = 0; hi = 0; return; }
    auto at = [&](int k) { return fma((double)(jb + k), dnu, numin) - nu; };
    const double off = (nu - numin) * inv_dnu - (double)jb, w = hw * inv_dnu;
    int l = (int)fmin(fmax(off - w, 0.0), (double)n);
    while (l > 0 && at(l - 1) > -hw) --l;
    while (l < n && !(at(l) > -hw)) ++l;
    int h = (int)fmin(fmax(off + w, 0.0), (double)n);
    while (h > 0 && !(at(h - 1) < hw)) --h;
    while (h < n && at(h) < hw) ++h;
    lo = l;
    hi = max(h, l);
}

// Chebyshev coefficient m (lane m < 20) of the node values F: T_m(u_k) =
// cos(m (2k + 1) pi / 40), cosv[j] = cos(j pi / 40).  Nodes k and 19 - k share a
// cosine up to its sign, and a middle value is taken off first: half the terms,
// and smaller ones.
__device__ __forceinline__ double cheb_coef64(const double *F, const double *cosv, int m) {
    const double base = F[kFN64 / 2], sg = m & 1 ? -1.0 : 1.0;
    double c = 0.0;
    int j = m;
#pragma unroll
    for (int k = 0; k < kFN64 / 2; ++k) {
        c = fma(fma(sg, F[kFN64 - 1 - k] - base, F[k] - base), cosv[j], c);
        j += 2 * m;
        j -= j >= 4 * kFN64 ? 4 * kFN64 : 0;
    }
    return m == 0 ? fma(1.0 / (double)kFN64, c, base) : 2.0 / (double)kFN64 * c;
}

// Adds g T_m(u), m = 0..19, to f.
__device__ __forceinline__ void add_moments20(double g, double u, double (&f)[kFN64]) {
    double p = g, c = g * u;
    const double u2 = 2.0 * u;
    f[0] += p;
    f[1] += c;
#pragma unroll
    for (int m = 2; m < kFN64; ++m) {
        const double n = fma(u2, c, -p);
        f[m] += n;
        p = c;
        c = n;
    }
}

// Node weight k from Chebyshev moments M: G_k = (M_0 + 2 sum M_m T_m(u_k)) / 20.
__device__ __forceinline__ double node_weight(const double *M, const double *cosv, int k) {
    double s = 0.0;
    int j = 2 * k + 1;
    const int step = j;
    for (int m = 1; m < kFN64; ++m) {
        s = fma(M[m], cosv[j], s);
        j += step;
        j -= j >= 4 * kFN64 ? 4 * kFN64 : 0;
    }
    return fma(2.0, s, M[0]) / (double)kFN64;
}

__device__ __forceinline__ double cheb_sum64(const double *c, double u) {
    double b1 = 0.0, b2 = 0.0;
    const double u2 = 2.0 * u;
#pragma unroll
    for (int m = kFN64 - 1; m >= 1; --m) {
        const double b0 = fma(u2, b1, c[m] - b2);
        b2 = b1;
        b1 = b0;
    }
    return fma(u, b1, c[0] - b2);
}

// ---------------------------------------------------------------------------
// Line core, x^2 + y^2 < 100: the midpoint rule for
//   w(x + iy) = (i/pi) int e^{-(x+s)^2} / (iy - s) ds
// on s = (k + 1/2) h (nodes that move with x, so the pole at s = iy is never
// near one), plus that pole's residue (Chiarella & Reichel 1968, Hunter &
// Regan 1972):
//   Re w = (h y/pi) sum_s e^{-(x+s)^2} / (s^2 + y^2)
//          + 2 e^{y^2-x^2} cos(2xy) / (1 + e^{2 pi y/h})     (y < pi/h)
// With x = (n0 + 1/2) h + d, |d| <= h/2, the 24 nodes that count have
// exponents -(d + m h)^2, m = -11..12: e^{-d^2} times a polynomial in
// e^{-2hd} whose coefficients are the constants e^{-h^2 m^2} and the line's
// table 1/(s^2 + y^2) at s = (n0 - m + 1/2) h.  h = 0.5178 leaves
// e^{-pi^2/h^2} = 1e-16 of the integral; relative error of Re w <= 5e-15
// against 50-digit values for 0 <= y < 10, tiny y and the far Doppler wing
// included (every term of the sum is positive).
// One exponential, one cosine and 24 table reads replace the 40 reciprocals
// and 4 exponentials of the Algorithm 916 series that a separate pass took
// (2.35e6 lines, 7e6 points at 10 bar: that pass 31 ms, the whole sum 39.9 ms,
// now 15.8; 1e5 lines, 3e6 points: 900 -> 497 us).
// ---------------------------------------------------------------------------
constexpr double kHC = 0.5178;
constexpr int kCLo = 11, kCHi = 12;               // m = -kCLo .. kCHi
constexpr int kCTab = 19 + kCLo + kCHi + 1;       // n0 <= 19
constexpr double kPiHC = 6.0671932282537524;      // pi / h
// e^{-h^2 m^2}
constexpr double kCE[kCHi + 1] = {
    1, 0.76481841449861865, 0.34216323515981589, 0.089541635567738392, 0.013706714729223335,
    0.0012273216551150678, 6.428358545165617e-05, 1.9695112154195025e-06, 3.5296650648060179e-08,
    3.7002000654827686e-10, 2.2689952580918315e-12, 8.1387674929739835e-15, 1.7076559162725319e-17};

// cos(t), 0 <= t <= 130, to ~1e-16 absolute: t = n pi + v in two parts, the
// Taylor series in v^2 (|v| <= pi/2; first term left out < 2e-17).
__device__ __forceinline__ double cos_bounded(double t) {
    constexpr double c[12] = {1.0, -1.0 / 2, 1.0 / 24, -1.0 / 720, 1.0 / 40320, -1.0 / 3628800,
                              1.0 / 479001600, -1.0 / 87178291200.0, 1.0 / 20922789888000.0,
                              -1.0 / 6402373705728000.0, 1.0 / 2432902008176640000.0,
                              -1.0 / 1124000727777607680000.0};
    const double n = rint(t * local_const(0.31830988618379067));
    double v = fma(-n, local_const(3.1415926535897931), t);
    v = fma(-n, local_const(1.2246467991473532e-16), v);
    const double w = v * v;
    double s = local_const(c[11]);
#pragma unroll
    for (int k = 10; k >= 1; --k) s = fma(s, w, local_const(c[k]));
    s = fma(s, w, 1.0);
    return ((int)n & 1) ? -s : s;
}

// Factor of e^{-x^2} cos(2xy) in sqrt(pi) Re w's pole term, per line.
__device__ __forceinline__ double core_pole(double y) {
    if (!(y < kPiHC)) return 0.0;
    const double b = y * (2.0 * kPiHC - y);          // 2 pi y/h - y^2 >= 0
    return 2.0 * exp_neg(b) / (1.0 + exp_neg(2.0 * kPiHC * y));
}

// The line's table, lane l < kCTab: 1/(s^2 + y^2), s = (l - kCHi + 1/2) h.
__device__ __forceinline__ void core_table(double *tab, double y2) {
    const int lane = threadIdx.x & 63;
    const double s = ((double)(lane - kCHi) + 0.5) * kHC;
    wave_lds_sync();
    if (lane < kCTab) tab[lane] = rcp64(fma(s, s, y2));
    wave_lds_sync();
}

// sqrt(pi) times the profile, times S: G h/2 e^{-d^2} (polynomial) + Apf
// e^{-x^2} cos(2xy), for |x| <= 10.
__device__ __forceinline__ double core_value(double x, double y, double G, double Apf,
                                             const double *tab) {
    const double ax = fmin(fabs(x), 10.0);
    const int n0 = (int)(ax * (1.0 / kHC));
    const double d = fma(-((double)n0 + 0.5), kHC, ax);
    const double *tb = tab + n0;
    const double r = exp_small(-2.0 * kHC * d), ri = rcp64(r);
    double P = 0.0, Q = 0.0;
#pragma unroll
    for (int m = kCHi; m >= 0; --m) {
        const double ce = local_const(kCE[m]);
        P = fma(P, r, ce * tb[kCHi - m]);
        if (m > 0 && m <= kCLo) Q = fma(Q, ri, ce * tb[kCHi + m]);
    }
    double v = (0.5 * kHC) * G * exp_small(-d * d) * fma(Q, ri, P);
    if (Apf != 0.0) v = fma(Apf * exp_neg(ax * ax), cos_bounded(2.0 * ax * y), v);
    return v;
}

// Binned Gaussian cell average of exp(-t^2)/sqrt(pi) times vb:
// (erf(x + h) - erf(x - h)) / 2 with h = vb/2, from the side away from the
// centre.
__device__ __forceinline__ double binned_gauss(double x, double h) {
    return x >= 0.0 ? 0.5 * (erfc(x - h) - erfc(x + h)) : 0.5 * (erfc(-x - h) - erfc(-x + h));
}

// Point-by-point part of one line on the wave's points: per 64-point segment
// 2 bits of code, 1: x^2 + y^2 >= 1e4 at all its points (4 nodes), 2: >= 100
// (8 nodes), 3: some points lie in the line core.
template <class P, int PPT, class Args>
__device__ __forceinline__ void add_points(const Args &a, uint32_t code, double nu, double ia,
                                           double y, double G, double Apf, double pl, int lo,
                                           int hi, bool full, double jd, double (&acc)[PPT],
                                           double *tab) {
    const int lane = threadIdx.x & 63;
    const double y2 = y * y, numin = a.numin, dnu = a.dnu;
    if (P::PROFILE == 1 && code & (code >> 1) & 0x55555555u) core_table(tab, y2);
    for (int k = 0; code != 0; ++k, code >>= 2) {
        const int c = code & 3;
        if (c == 0) continue;
        const double xj = fma(jd + (double)(64 * k), dnu, numin);
        const double dd = xj - nu;
        const double x = dd * ia;
        const double x2 = x * x;
        const double r2 = fma(x, x, y2);
        double v = 0.0, num, den;
        if (P::PROFILE == 0) {
        } else if (P::PROFILE == 2) {
            v = G / r2;
        } else if (P::PROFILE == 3) {
            v = G * exp_neg(fmin(x2, 800.0));
        } else if (P::PROFILE == 4) {
            const double vb = dnu * ia;
            v = G / vb * binned_gauss(x, 0.5 * vb);
        } else if (c == 1) {
            gh_frac(GH<2>(), x2, r2, num, den);
            v = G * (num * rcp64(den));
        } else if (c == 2 || __ballot(r2 >= kRB64) != 0ull) {
            gh_frac(GH<4>(), x2, r2, num, den);
            v = G * (num * rcp64(den));
        }
        if (P::PROFILE == 1 && c == 3) {
            const double w = core_value(x, y, G, Apf, tab);
            v = r2 < kRB64 ? w : v;
        }
        if constexpr (P::CHI) {
            if (xj > a.chi.lo && xj < a.chi.hi)
                v *= exp_neg(fmin(chi_exponent(a.chi, fabs(dd)), 800.0)) * (xj / nu);
        }
        // (plinths alone: a line that covers the wave is in the constants)
        if (P::PLINTH && (P::PROFILE != 0 || !full)) v -= pl;
        if (!full) {
            const int j = lane + 64 * k;
            v = (j >= lo && j < hi) ? v : 0.0;
        }
        // one copy of the code above for all segments: acc is a register
        // array, so the segment's sum is picked by uniform branches
#pragma unroll
        for (int q = 0; q < PPT; ++q)
            if (q == k) acc[q] += v;
    }
}

// A line that covers the wave's 64 PPT points with one wing formula (N: 0, Lorentz
// less the plinth, 1, the asymptotic series, for x^2 + y^2 >= 1e6, 2 for >= 1e4, 4 for >= 100): a lane's
// points side by side, so that their reciprocals' chains overlap.
template <int N, int PPT, class XAt>
__device__ __forceinline__ void add_wing(const XAt &x_at, double nu, double ia, double y, double G,
                                         double pl, double (&acc)[PPT]) {
    const double y2 = y * y;
    const GH<N == 4 ? 4 : 2> gh;
    // (series: G is S y / pi, as in add_nodes)
    if (N == 1) G *= 0.5 * kPi * kISqrtPi;
    const double p2 = fma(-2.0, y2, 3.75), p3 = -15.0 * y2, p4 = 12.0 * y2 * y2;
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        if (k > 0 && k % 4 == 0) __builtin_amdgcn_sched_barrier(0);   // (16 at once: spills)
        const double x = (x_at(k) - nu) * ia;
        const double r2 = fma(x, x, y2);
        if (N == 0) {
            acc[k] += G / r2 - pl;
        } else if (N == 1) {
            const double q = rcp64(r2);
            acc[k] += fma(G * q, fma(fma(fma(fma(p4, q, p3), q, p2), q, 1.5), q, 1.0), -pl);
        } else {
            double num, den;
            gh_frac(gh, x * x, r2, num, den);
            acc[k] += fma(G, num * rcp64(den), -pl);
        }
    }
}

// The wave's part of a tile.
struct WavePoints {
    int64_t jw;                 // first point
    int nw;                     // points
    double xwf, jd, inv_dnu;    // centre of the first, this lane's index, 1/dnu
};

// Up to 64 lines point by point: one line per lane (i: its index, -1: none) finds
// its window and formulas on the wave's points, then the wave takes them in turn.
template <int PPT, class P, class Args, class XAt>
__device__ __forceinline__ void add_lines(const Args &a, int64_t i, const WavePoints &w,
                                          const XAt &x_at, double (&acc)[PPT], double *tab) {
    constexpr int WP = 64 * PPT;
    const int64_t jw = w.jw;
    const int nw = w.nw;
    const double xwf = w.xwf, jd = w.jd, inv_dnu = w.inv_dnu;
    uint32_t code = 0;
    int lo = 0, hi = 0;
    double nu = 0.0, ia = 1.0, y = 1.0, G = 0.0, Apf = 0.0, pl = 0.0;
    bool far = false;                            // x^2 + y^2 >= 1e6 at all points
    if (i >= 0) {
        nu = a.nu[i];
        const double hw = a.hw[i], S = a.S[i];
        y = a.y[i];
        ia = a.ia[i];
        clip_window(nu, hw, a.numin, a.dnu, inv_dnu, jw, nw, lo, hi);
        if (lo < hi) {
            G = line_factor<P>(S, y);
            if constexpr (P::PLINTH) pl = a.pl[i];
            if constexpr (P::PROFILE == 1) {
                // conservative point intervals with x^2 + y^2 < 100, 1e4
                const float vb = (float)(a.dnu * ia), fy2 = (float)(y * y);
                const float cen = (float)((nu - xwf) * inv_dnu);
                const float r1 = sqrtf(fmaxf(1.0002e2f - fy2, 0.0f)) / vb;
                const float r2 = sqrtf(fmaxf(1.0002e4f - fy2, 0.0f)) / vb;
                const float mg = 2.0f + 1.0e-5f * fabsf(cen);
                const bool in1 = fy2 < 1.0002e2f, in2 = fy2 < 1.0002e4f;
                if constexpr (P::WHOLE) {
                    const float r3 = sqrtf(fmaxf(1.0002e6f - fy2, 0.0f)) / vb;
                    far = !(fy2 < 1.0002e6f && cen - r3 - mg <= (float)(WP - 1) &&
                            cen + r3 + mg >= 0.0f) && fy2 < 1.0e12f;
                }
#pragma unroll
                for (int k = 0; k < PPT; ++k) {
                    const int s0 = 64 * k, s1 = s0 + 63;
                    if (lo > s1 || hi <= s0) continue;
                    const bool c3 = in1 && cen - r1 - mg <= (float)s1 && cen + r1 + mg >= (float)s0;
                    const bool c2 = in2 && cen - r2 - mg <= (float)s1 && cen + r2 + mg >= (float)s0;
                    code |= (c3 ? 3u : c2 ? 2u : 1u) << (2 * k);
                }
                if (code & (code >> 1) & 0x55555555u) Apf = S * kISqrtPi * core_pole(y);
            } else {
                // segments that the window touches; a compact profile's
                // only where it is not zero, unless a plinth is there
                int l = lo, h = hi;
                const bool part = P::PROFILE == 0 || (P::PLINTH && pl != 0.0);
                if (P::COMPACT && !part && fabs(S) < 1.0e300) {
                    const double off = (nu - xwf) * inv_dnu;
                    const double w = kDopplerEnd / ia * inv_dnu + 2.0;
                    l = max(lo, (int)fmin(fmax(off - w, 0.0), (double)nw));
                    h = min(hi, (int)fmin(fmax(off + w, 0.0), (double)nw));
                }
                if (P::PROFILE != 0 || part)
#pragma unroll
                    for (int k = 0; k < PPT; ++k)
                        if (l < 64 * k + 64 && h > 64 * k && l < h) code |= 1u << (2 * k);
            }
        }
    }
    unsigned long long m = __ballot(code != 0);
    if constexpr (P::WHOLE) {
        // lines of one formula over the wave, in a loop of its own each:
        // merged, every line copies the sums between its paths
        constexpr uint32_t ones = 0x55555555u & (uint32_t)((1ull << (2 * PPT)) - 1);
        const bool whole = lo == 0 && hi == WP;
        auto wings = [&](auto formula, bool these) {
            unsigned long long q = __ballot(these);
            m &= ~q;
            while (q) {
                const int b = __builtin_ctzll(q);
                q &= q - 1ull;
                add_wing<formula, PPT>(x_at, lane_f64(nu, b), lane_f64(ia, b),
                                       lane_f64(y, b), lane_f64(G, b),
                                       P::PLINTH ? lane_f64(pl, b) : 0.0, acc);
            }
        };
        if constexpr (P::PROFILE == 2) {
            wings(std::integral_constant<int, 0>{}, whole && code == ones);
        } else {
            wings(std::integral_constant<int, 1>{}, whole && code == ones && far);
            wings(std::integral_constant<int, 2>{}, whole && code == ones && !far);
            wings(std::integral_constant<int, 4>{}, whole && code == 2 * ones);
        }
    }
    while (m) {
        const int b = __builtin_ctzll(m);
        m &= m - 1ull;
        const int slo = __builtin_amdgcn_readlane(lo, b), shi = __builtin_amdgcn_readlane(hi, b);
        const uint32_t scode = (uint32_t)__builtin_amdgcn_readlane((int)code, b);
        add_points<P, PPT>(a, scode,
                           lane_f64(nu, b), lane_f64(ia, b), lane_f64(y, b), lane_f64(G, b),
                           P::PROFILE == 1 ? lane_f64(Apf, b) : 0.0,
                           P::PLINTH ? lane_f64(pl, b) : 0.0, slo, shi,
                           slo == 0 && shi == nw, jd, acc, tab);
    }
}

// Writes the wave's sums.
template <int PPT, class P, class Args, class XAt>
__device__ __forceinline__ void store_points(const Args &a, const WavePoints &w, const XAt &x_at,
                                             const double (&acc)[PPT]) {
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const int64_t j = w.jw + (threadIdx.x & 63) + 64 * k;
        if constexpr (P::CHI) {
            const double x = x_at(k);
            if (a.side != 0 && (x > a.lo && x < a.hi) != (a.side > 0)) continue;
        }
        if (j < a.nx) a.K[j] = a.accumulate ? a.K[j] + acc[k] : a.kmin + acc[k];
    }
}

template <int PPT, class P, class Args>
__device__ __forceinline__ void tile_f64(const Args &a, int64_t tile, Far64LDS *sh) {
    constexpr int W = kThreads * PPT, WP = 64 * PPT;
    constexpr bool kNodes = P::WINGS && !P::EXACT;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t j0 = tile * W, jw = j0 + wave * WP;
    const int Wv = (int)min((int64_t)W, a.nx - j0);                    // valid points
    const int nw = max(0, min(WP, Wv - wave * WP));
    const double inv_dnu = 1.0 / a.dnu;
    // tile and wave centres and half widths (of their valid points)
    const double xfirst = fma((double)j0, a.dnu, a.numin);
    const double xlast = fma((double)(j0 + Wv - 1), a.dnu, a.numin);
    const double hW = fmax(0.5 * (double)(Wv - 1), 0.5) * a.dnu;
    const double xc = fma((double)j0 + 0.5 * (double)(Wv - 1), a.dnu, a.numin);
    const double xwf = fma((double)jw, a.dnu, a.numin);
    const double hw_w = fmax(0.5 * (double)(nw - 1), 0.5) * a.dnu;
    const double xcw = fma((double)jw + 0.5 * (double)max(nw - 1, 0), a.dnu, a.numin);
    const double jd = (double)(jw + lane);        // this lane's first point
    double acc[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) acc[k] = 0.0;
    // this lane's points, kept where most of the work is theirs
    double xj[P::EXACT ? PPT : 1];
    auto x_of = [&](int k) { return fma(jd + (double)(64 * k), a.dnu, a.numin); };
    auto x_at = [&](int k) { return P::EXACT ? xj[P::EXACT ? k : 0] : x_of(k); };
    if constexpr (P::EXACT) {
#pragma unroll
        for (int k = 0; k < PPT; ++k) xj[k] = x_of(k);
    }
    // line range of the tile: waves 0 and 1 search one end each
    auto clear = [&]() {
        if (t < 4 * kFN64) sh->cosv[t] = cos40(t);
        if (lane < kFN64) { sh->F[wave][lane] = 0.0; sh->wF[wave][lane] = 0.0; }
    };
    if constexpr (!P::SPARSE) clear();
    if (wave < 2) {
        const double R = a.radius[0];
        int64_t b = 0;
        if (R > 0.0 && a.nl > 0)
            b = wave == 0 ? wave_bound<true>(a.key, a.nl, xfirst - R)
                          : wave_bound<false>(a.key, a.nl, xlast + R);
        if (lane == 0) sh->range[wave] = b;
    }
    __syncthreads();
    const int64_t first = sh->range[0], last = sh->range[1];
    const WavePoints w = {jw, nw, xwf, jd, inv_dnu};
    if constexpr (P::SPARSE) {
        if (last - first <= kFewLines) {
            if (nw == 0) return;
            if (first < last)
                add_lines<PPT, P>(a, lane < last - first ? first + lane : -1, w, x_at, acc,
                                  sh->tab[wave]);
            store_points<PPT, P>(a, w, x_at, acc);
            return;
        }
        clear();                                 // (barriers follow before its readers)
    }
    bool any_far = false, any_wave = false;
    // plinths alone: those of lines that cover the tile, the wave
    constexpr bool kConst = P::PLINTH && P::PROFILE == 0;
    double cst = 0.0, wcst = 0.0;
    for (int64_t r0 = first; r0 < last; r0 += kRound64) {
        const int nr = (int)min((int64_t)kRound64, last - r0);
        // tile level: one line per lane; near lines listed per wave
        int cnt = 0;
        {
            double f[kFN64];
#pragma unroll
            for (int k = 0; k < kFN64; ++k) f[k] = 0.0;
            bool used = false;
            for (int s0 = 0; s0 < nr; s0 += kThreads) {
                const int e = s0 + t;
                bool near = false;
                int cls = 0;
                double D = 1.0, ia = 1.0, y2 = 1.0, G = 0.0, pl = 0.0;
                ChiPiece chi;
                if (e < nr) {
                    const int64_t i = r0 + e;
                    // (all loads at once: one wait on memory, not three)
                    const double nu = a.nu[i], hw = a.hw[i];
                    double y = 0.0, S = 0.0;
                    if constexpr (kNodes || P::COMPACT) { ia = a.ia[i]; S = a.S[i]; }
                    if constexpr (kNodes) y = a.y[i];
                    const double dl = xfirst - nu, dh = xlast - nu;
                    near = hw > 0.0 && dl < hw && dh > -hw;
                    const bool full = dl > -hw && dl < hw && dh > -hw && dh < hw;
                    D = xc - nu;
                    if constexpr (P::PLINTH) {
                        if (near) pl = a.pl[i];
                    }
                    if constexpr (kConst) {
                        if (near && full) cst -= pl;
                        near = near && !full;
                    } else if (P::COMPACT) {
                        if (near && !(P::PLINTH && pl != 0.0) && fabs(S) < 1.0e300)
                            near = (fabs(D) - hW - a.dnu) * ia <= kDopplerEnd;
                    } else if (kNodes && near && full && fabs(D) >= kFarRatio64 * hW) {
                        y2 = y * y;
                        G = line_factor<P>(S, y);
                        cls = far_class64<P>(D, hW, ia, y2, G);
                        if constexpr (P::CHI) {
                            if (cls && !chi_piece(a.chi, xfirst, xlast, nu, D, hW, chi)) cls = 0;
                        }
                        near = cls == 0;
                    }
                }
                if constexpr (kNodes) {
                    used |= __ballot(cls != 0) != 0ull;
                    add_far_lines<P>(cls, D, hW, ia, y2, G, pl, chi, f);
                }
                const unsigned long long m = __ballot(near);
                if (near)
                    sh->list[wave][cnt + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)e;
                cnt += __popcll(m);
            }
            if (used) { add_node_totals(f, sh->F[wave]); any_far = true; }
        }
        if (lane == 0) sh->cnt[wave] = cnt;
        __syncthreads();
        // near lines of all waves, in chunks of 64, one line per lane
        int cum[kWaves + 1];
        cum[0] = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) cum[w + 1] = cum[w] + sh->cnt[w];
        const int total = nw > 0 ? cum[kWaves] : 0;
        auto line_at = [&](int e) {
            int w = 0, c = 0;
#pragma unroll
            for (int q = 1; q < kWaves; ++q)
                if (e >= cum[q]) { w = q; c = cum[q]; }
            return r0 + sh->list[w][e - c];
        };
        // wave level (a loop of its own: its node sums and the point loop's
        // values do not fit the registers together)
        if constexpr (kNodes || kConst) {
            double f[kFN64];
#pragma unroll
            for (int k = 0; k < kFN64; ++k) f[k] = 0.0;
            bool used = false;
            const double xwl = fma((double)(jw + nw - 1), a.dnu, a.numin);
            for (int c0 = 0; c0 < total; c0 += 64) {
                int cls = 0;
                double D = 1.0, ia = 1.0, y2 = 1.0, G = 0.0, pl = 0.0;
                ChiPiece chi;
                if (c0 + lane < total) {
                    const int64_t i = line_at(c0 + lane);
                    const double nu = a.nu[i], hw = a.hw[i];
                    double y = 0.0, S = 0.0;
                    if constexpr (kNodes) { ia = a.ia[i]; S = a.S[i]; y = a.y[i]; }
                    const double dl = xwf - nu, dh = xwl - nu;
                    D = xcw - nu;
                    const bool full = dl > -hw && dl < hw && dh > -hw && dh < hw;
                    if constexpr (kConst) {
                        const double el = xfirst - nu, eh = xlast - nu;
                        if (full && !(el > -hw && el < hw && eh > -hw && eh < hw)) wcst -= a.pl[i];
                    }
                    if (kNodes && full && fabs(D) >= kFarRatio64 * hw_w) {
                        y2 = y * y;
                        G = line_factor<P>(S, y);
                        if constexpr (P::PLINTH) pl = a.pl[i];
                        cls = far_class64<P>(D, hw_w, ia, y2, G);
                        if constexpr (P::CHI) {
                            if (cls && !chi_piece(a.chi, xwf, xwl, nu, D, hw_w, chi)) cls = 0;
                        }
                    }
                }
                unsigned long long wm = __ballot(cls != 0);
                if (__popcll(wm) >= wave_min_lines(PPT)) {
                    add_far_lines<P>(cls, D, hw_w, ia, y2, G, pl, chi, f);
                    used = true;
                } else wm = 0ull;
                if (lane == 0) sh->taken[wave][c0 >> 6] = wm;
            }
            if (used) { add_node_totals(f, sh->wF[wave]); any_wave = true; }
        }
        wave_lds_sync();
        // the rest point by point
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int e = c0 + lane;
            const bool mine =
                e < total && !((kNodes || kConst) && (sh->taken[wave][c0 >> 6] >> lane) & 1ull);
            add_lines<PPT, P>(a, mine ? line_at(e) : -1, w, x_at, acc, sh->tab[wave]);
        }
        __syncthreads();      // the lists are free for the next round
    }
    // node sums -> one series per wave.  any_far differs between waves: the
    // tile's totals are taken whenever any wave has some.
    if (kConst) {
        const double c = wave_total64(cst);
        if (lane == 0) sh->cst[wave] = c;
    }
    const bool tile_far = __syncthreads_or(any_far) != 0;
    if (nw == 0) return;
    if (kConst) {
        double c = wave_total64(wcst);
#pragma unroll
        for (int w = 0; w < kWaves; ++w) c += sh->cst[w];
#pragma unroll
        for (int k = 0; k < PPT; ++k) acc[k] += c;
    }
    if (tile_far || any_wave) {
        double *c = sh->c[wave], *wF = sh->wF[wave];
        if (tile_far) {
            if (lane < kFN64) {
                double s = 0.0;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) s += sh->F[w][lane];
                c[lane] = s;
            }
            wave_lds_sync();
            const double cm = lane < kFN64 ? cheb_coef64(c, sh->cosv, lane) : 0.0;
            wave_lds_sync();
            if (lane < kFN64) c[lane] = cm;
            wave_lds_sync();
            if (lane < kFN64) {
                wF[lane] += cheb_sum64(c, (fma(node_u(lane), hw_w, xcw - xc)) / hW);
            }
            wave_lds_sync();
        }
        const double cm = lane < kFN64 ? cheb_coef64(wF, sh->cosv, lane) : 0.0;
        wave_lds_sync();
        if (lane < kFN64) c[lane] = cm;
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < PPT; ++k)
            acc[k] += cheb_sum64(c, (fma(jd + (double)(64 * k), a.dnu, a.numin) - xcw) / hw_w);
    }
    store_points<PPT, P>(a, w, x_at, acc);
}

}  // namespace hk
