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
// a double pole) interpolates to 5e-15 of its value, largest at the tile end
// nearest the line; everything else is FP64 rounding, as in the pair sum.
// The nodes and the points are placed relative to the tile centre, so the
// rounding of x_j = fma(j, dnu, numin) enters the far field exactly as it
// enters a pair.
//
// What bounds it: FP64 vector instructions.  At 1e5 lines, 3e6 points, cut
// 100 cm^-1 a line has 2e4 pairs in its window; it takes 20 node values in
// each of ~17 tiles, 20 in ~9 waves and ~13 instructions' worth of 64
// points -- 30 times fewer evaluations than pairs.
#pragma once
#include "hk_device.h"
#include "hk_tiles.h"

namespace hk {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

constexpr int kFN64 = 20;                 // Chebyshev-Gauss nodes
constexpr double kFarRatio64 = 3.25;
// Largest x^2 + y^2 of a far line: keeps the products of the 8-node rule
// (~ r2^16 for a pair of nodes) in range.
constexpr double kFarMaxR2 = 1.0e18;
// cos(pi (k + 1/2) / 20), k = 0..9; node 19 - k is its negative
constexpr double kU64[kFN64 / 2] = {0.99691733373312796, 0.97236992039767667, 0.92387953251128674,
                                    0.85264016435409218, 0.76040596560003093, 0.64944804833018377,
                                    0.52249856471594880, 0.38268343236508984, 0.23344536385590542,
                                    0.078459095727844999};
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
    double cosv[4 * kFN64];                     // cos(j pi / 40)
    int cnt[kWaves];
    int64_t range[2];
};

// A uniform constant the compiler cannot hoist: the unrolled node loops use
// dozens of FP64 literals, and kept in scalar registers across the tile loop
// they spill.
__device__ __forceinline__ double local_const(double v) {
    asm volatile("" : "+s"(v));
    return v;
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

// Far class of a line for an interval of half width `half` whose centre lies
// D from the line centre [cm^-1]: 0 = not far, else the wing formula its
// nearest point allows (1 series, 2 four nodes, 3 eight nodes).
__device__ __forceinline__ int far_class64(double D, double half, double ia, double y2, double G) {
    const double d = fabs(D);
    const double xn = (d - half) * ia, xf = (d + half) * ia;
    const double rn = fma(xn, xn, y2), rf = fma(xf, xf, y2);
    const bool ok = d >= kFarRatio64 * half && rn >= kRB64 && rf < kFarMaxR2 &&
                    fabs(G) < 1.0e300;
    return !ok ? 0 : rn >= kRF64 ? 1 : rn >= kRM64 ? 2 : 3;
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
// reciprocal.  g = 2 S y / pi^1.5 (0 for a lane without a line).
template <int CLASS>
__device__ __forceinline__ void add_nodes(double D, double half, double ia, double y2, double g,
                                          double (&f)[kFN64]) {
    const double xc = D * ia, h = half * ia;
    double p2 = 0.0, p3 = 0.0, p4 = 0.0;
    if (CLASS == 1) {
        p2 = fma(-2.0, y2, 3.75); p3 = -15.0 * y2; p4 = 12.0 * y2 * y2;
        g *= 0.5 * kPi * kISqrtPi;      // S y / pi
    }
    const GH<CLASS == 3 ? 4 : 2> gh;
#pragma unroll
    for (int k = 0; k < kFN64 / 2; ++k) {
        __builtin_amdgcn_sched_barrier(0);   // (pairs interleaved: spills)
        const double u = local_const(kU64[k]);
        const double xa = fma(u, h, xc), xb = fma(-u, h, xc);
        const double a2 = xa * xa, b2 = xb * xb;
        const double ra = a2 + y2, rb = b2 + y2;
        if (CLASS == 1) {
            const double q = rcp64(ra * rb), ia1 = q * rb, ib1 = q * ra;
            const double va = fma(fma(fma(fma(p4, ia1, p3), ia1, p2), ia1, 1.5), ia1, 1.0);
            const double vb = fma(fma(fma(fma(p4, ib1, p3), ib1, p2), ib1, 1.5), ib1, 1.0);
            f[k] = fma(g * ia1, va, f[k]);
            f[kFN64 - 1 - k] = fma(g * ib1, vb, f[kFN64 - 1 - k]);
        } else {
            double na, da, nb, db;
            gh_frac(gh, a2, ra, na, da);
            gh_frac(gh, b2, rb, nb, db);
            // (g last: strengths far below 1e-100 must not meet the products)
            const double q = rcp64(da * db);
            f[k] = fma(g, na * db * q, f[k]);
            f[kFN64 - 1 - k] = fma(g, nb * da * q, f[kFN64 - 1 - k]);
        }
    }
}

// The lanes with cls != 0 add their lines' node values; the whole wave takes
// the formula of the line nearest its interval (valid farther out too).
__device__ __forceinline__ void add_far_lines(int cls, double D, double half, double ia, double y2,
                                              double G, double (&f)[kFN64]) {
    if (__ballot(cls != 0) == 0ull) return;
    if (cls == 0) { D = 1.0; half = 0.0; ia = 1.0e4; y2 = 0.0; G = 0.0; }
    if (__ballot(cls == 3)) add_nodes<3>(D, half, ia, y2, G, f);
    else if (__ballot(cls == 2)) add_nodes<2>(D, half, ia, y2, G, f);
    else add_nodes<1>(D, half, ia, y2, G, f);
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
// cos(m (2k + 1) pi / 40), cosv[j] = cos(j pi / 40).
__device__ __forceinline__ double cheb_coef64(const double *F, const double *cosv, int m) {
    double c = 0.0;
    int j = m;
    for (int k = 0; k < kFN64; ++k) {
        c = fma(F[k], cosv[j], c);
        j += 2 * m;
        j -= j >= 4 * kFN64 ? 4 * kFN64 : 0;
    }
    return (m == 0 ? 1.0 : 2.0) / (double)kFN64 * c;
}

// Orders a wave's own LDS writes before its later reads of them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
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

__device__ __forceinline__ double lane_f64(double v, int b) {
    const long long x = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)x, b);
    const unsigned hi = __builtin_amdgcn_readlane((int)(x >> 32), b);
    return __longlong_as_double(((long long)hi << 32) | lo);
}

// Point-by-point part of one line on the wave's points: per 64-point segment
// 2 bits of code, 1: x^2 + y^2 >= 1e4 at all its points (4 nodes), 2: >= 100
// (8 nodes), 3: some points lie in the line core (skipped here; the line-core
// pass adds them).
template <int PPT>
__device__ __forceinline__ void add_points(uint32_t code, double nu, double ia, double y2, double G,
                                           int lo, int hi, bool full, const double (&xj)[PPT],
                                           double (&acc)[PPT]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const int c = (code >> (2 * k)) & 3;
        if (c == 0) continue;
        const double x = (xj[k] - nu) * ia;
        const double x2 = x * x;
        double v;
        if (c == 1) {
            double num, den;
            gh_frac(GH<2>(), x2, x2 + y2, num, den);
            v = G * (num * rcp64(den));
        } else {
            const double r2 = fma(x, x, y2);
            double num, den;
            gh_frac(GH<4>(), x2, r2, num, den);
            v = G * (num * rcp64(den));
            if (c == 3) v = r2 >= kRB64 ? v : 0.0;
        }
        if (!full) {
            const int j = lane + 64 * k;
            v = (j >= lo && j < hi) ? v : 0.0;
        }
        acc[k] += v;
    }
}

template <int PPT, class Args>
__device__ __forceinline__ void tile_f64(const Args &a, int64_t tile, Far64LDS *sh) {
    constexpr int W = kThreads * PPT, WP = 64 * PPT;
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
    double xj[PPT], acc[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        xj[k] = fma((double)(jw + lane + 64 * k), a.dnu, a.numin);
        acc[k] = 0.0;
    }
    // line range of the tile: waves 0 and 1 search one end each
    if (t < 4 * kFN64) sh->cosv[t] = cospi((double)t / (2.0 * kFN64));
    if (lane < kFN64) { sh->F[wave][lane] = 0.0; sh->wF[wave][lane] = 0.0; }
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
    bool any_far = false, any_wave = false;
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
                double D = 1.0, ia = 1.0, y2 = 1.0, G = 0.0;
                if (e < nr) {
                    const int64_t i = r0 + e;
                    const double nu = a.nu[i], hw = a.hw[i];
                    const double dl = xfirst - nu, dh = xlast - nu;
                    near = hw > 0.0 && dl < hw && dh > -hw;
                    const bool full = dl > -hw && dl < hw && dh > -hw && dh < hw;
                    D = xc - nu;
                    if (a.far && near && full && fabs(D) >= kFarRatio64 * hW) {
                        const double y = a.y[i];
                        ia = a.ia[i];
                        y2 = y * y;
                        G = a.S[i] * y * (kISqrtPi * 2.0 / kPi);
                        cls = far_class64(D, hW, ia, y2, G);
                        near = cls == 0;
                    }
                }
                used |= __ballot(cls != 0) != 0ull;
                add_far_lines(cls, D, hW, ia, y2, G, f);
                const unsigned long long m = __ballot(near);
                if (near)
                    sh->list[wave][cnt + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)e;
                cnt += __popcll(m);
            }
            if (used) { add_node_totals(f, sh->F[wave]); any_far = true; }
        }
        if (lane == 0) sh->cnt[wave] = cnt;
        __syncthreads();
        // near lines of all waves, 64 at a time, one per lane
        int cum[kWaves + 1];
        cum[0] = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) cum[w + 1] = cum[w] + sh->cnt[w];
        const int total = nw > 0 ? cum[kWaves] : 0;
        double f[kFN64];
#pragma unroll
        for (int k = 0; k < kFN64; ++k) f[k] = 0.0;
        bool used = false;
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int e = c0 + lane;
            uint32_t code = 0;
            int lo = 0, hi = 0, cls = 0;
            double nu = 0.0, ia = 1.0, y2 = 1.0, G = 0.0, D = 1.0;
            if (e < total) {
                int w = 0;
#pragma unroll
                for (int q = 1; q < kWaves; ++q) w += e >= cum[q];
                const int64_t i = r0 + sh->list[w][e - (w == 0 ? 0 : w == 1 ? cum[1] : w == 2 ? cum[2] : cum[3])];
                nu = a.nu[i];
                const double hw = a.hw[i], y = a.y[i];
                ia = a.ia[i];
                y2 = y * y;
                G = a.S[i] * y * (kISqrtPi * 2.0 / kPi);
                clip_window(nu, hw, a.numin, a.dnu, inv_dnu, jw, nw, lo, hi);
                if (lo < hi) {
                    D = xcw - nu;
                    if (a.far && lo == 0 && hi == nw) cls = far_class64(D, hw_w, ia, y2, G);
                    // conservative point intervals with x^2 + y^2 < 100, 1e4
                    const float vb = (float)(a.dnu * ia), fy2 = (float)y2;
                    const float cen = (float)((nu - xwf) * inv_dnu);
                    const float r1 = sqrtf(fmaxf(1.0002e2f - fy2, 0.0f)) / vb;
                    const float r2 = sqrtf(fmaxf(1.0002e4f - fy2, 0.0f)) / vb;
                    const float mg = 2.0f + 1.0e-5f * fabsf(cen);
                    const bool in1 = fy2 < 1.0002e2f, in2 = fy2 < 1.0002e4f;
#pragma unroll
                    for (int k = 0; k < PPT; ++k) {
                        const int s0 = 64 * k, s1 = s0 + 63;
                        if (lo > s1 || hi <= s0) continue;
                        const bool c3 = in1 && cen - r1 - mg <= (float)s1 && cen + r1 + mg >= (float)s0;
                        const bool c2 = in2 && cen - r2 - mg <= (float)s1 && cen + r2 + mg >= (float)s0;
                        code |= (c3 ? 3u : c2 ? 2u : 1u) << (2 * k);
                    }
                }
            }
            const unsigned long long wm = __ballot(cls != 0);
            if (__popcll(wm) >= wave_min_lines(PPT)) {
                add_far_lines(cls, D, hw_w, ia, y2, G, f);
                used = true;
                if (cls) code = 0;
            }
            unsigned long long m = __ballot(code != 0);
            while (m) {
                const int b = __builtin_ctzll(m);
                m &= m - 1ull;
                const int slo = __builtin_amdgcn_readlane(lo, b), shi = __builtin_amdgcn_readlane(hi, b);
                add_points<PPT>((uint32_t)__builtin_amdgcn_readlane((int)code, b), lane_f64(nu, b),
                                lane_f64(ia, b), lane_f64(y2, b), lane_f64(G, b), slo, shi,
                                slo == 0 && shi == nw, xj, acc);
            }
        }
        if (used) { add_node_totals(f, sh->wF[wave]); any_wave = true; }
        __syncthreads();      // the lists are free for the next round
    }
    // node sums -> one series per wave.  any_far differs between waves: the
    // tile's totals are taken whenever any wave has some.
    const bool tile_far = __syncthreads_or(any_far) != 0;
    if (nw == 0) return;
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
                const double u = lane < kFN64 / 2 ? kU64[lane] : -kU64[kFN64 - 1 - lane];
                wF[lane] += cheb_sum64(c, (fma(u, hw_w, xcw - xc)) / hW);
            }
            wave_lds_sync();
        }
        const double cm = lane < kFN64 ? cheb_coef64(wF, sh->cosv, lane) : 0.0;
        wave_lds_sync();
        if (lane < kFN64) c[lane] = cm;
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < PPT; ++k) acc[k] += cheb_sum64(c, (xj[k] - xcw) / hw_w);
    }
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const int64_t j = jw + lane + 64 * k;
        if (j < a.nx) a.K[j] = a.accumulate ? a.K[j] + acc[k] : a.kmin + acc[k];
    }
}

}  // namespace hk
