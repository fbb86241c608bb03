// hk_adjoint.hip -- adjoint of the Voigt sum.
//
// For L = sum_j gK_j K_j with K_j = kmin + sum_i S_i Re w(x_ij, y_i)/sqrt(pi)
// (the forward sum of hk_voigt_accumulate) the line parameters (FP64, as
// hk_line_params) and the complex profile w on each line's cut window are
// recomputed -- nothing of the forward pass is stored:
//   dL/dS_i   = F_i  sum_j gK_j Re w / sqrt(pi)              (S = S_file)
//   dL/dvy_i  = S_i  sum_j gK_j dRe w/dy / sqrt(pi) * dy/dvy
//   dL/dT, dL/dP = sum_i S_i sum_j gK_j [Re w dlnS + dRe w/dx dx + dRe w/dy dy]
// with w'(z) = -2 z w + 2i/sqrt(pi):  dRe w/dx = -2 (x Re w - y Im w),
// dRe w/dy = 2 (x Im w + y Re w) - 2/sqrt(pi) for |z|^2 < 1e4, and from the
// asymptotic series of w' beyond (the identity cancels to ~eps |z|^2).  The
// partition function is held fixed.
//
// Per line four sums over its window are needed: of gK times Re w, dRe w/dy,
// dRe w/dx and x dRe w/dx.  They are the transpose of the forward sum, and its
// far field transposes with them: over an interval far from the line (or a
// wave's worth, or 64 points) the profile is the polynomial through its values
// f_k at the interval's 20 Chebyshev nodes, so
//   sum_j gK_j f(x_j) = sum_k f_k G_k,   G_k = sum_j gK_j l_k(x_j),
// with l_k the nodes' Lagrange polynomials.  A workgroup owns 256 consecutive
// lines, one per lane (64 of a short list, its waves sharing their work), and
// walks the 1024-point tiles (256 or 512 for short lists) that their windows
// reach: it forms the G_k of the tile, and of its four quarters and 16 segments where
// some line is near, and each lane evaluates its line at the nodes of the
// largest far interval; what is left (~4 segments a line) is summed point by
// point, 64 points at a time.  Tiles between two windows are passed over, and the
// windows of a short list that are few and short against their tiles are summed
// point by point throughout.
//
// What bounds it: FP64 vector instructions, about half of them the line cores.
// One wave per line over all points of its window took 13.3 ms for 3.3e5 lines
// on 1e6 points, cut 50 cm^-1 (3.3e9 pairs), this 2.14 (with 3 workgroups a CU
// for the registers, as the compiler chooses, 2.23).
#include <math.h>

#include <algorithm>

#include "hk_device.h"
#include "hk_internal.h"
#include "hk_voigt64.h"

namespace {

using namespace hk;

// A derivative of the narrowest line is a triple pole: at 3.5 half widths 20
// nodes leave 5e-15 of its largest value.
constexpr double kFarRatioAdj = 3.5;
constexpr int kAT = 256;                  // lines per workgroup
constexpr int kATile = 1024, kASub = 256, kASeg = 64;
constexpr int kASubs = kATile / kASub, kASegs = kATile / kASeg;

// Short lists: a line is summed by itself, 64 points of its window a step, where
// that takes at most this many steps per tile that a workgroup would walk.  With
// 0, 20, 40 and 80 (1e6 points): 500 lines of 1000 points 137, 31, 31, 31 us,
// 3000 of 5000 points 178, 175, 82, 82, 10000 of 5000 269, 271, 272, 210, 50000 of
// 5000 625, 628, 625, 750; on 1e5 points 10000 of 5000 166, 167, 167, 205.
// What counts is the average window, and the wave with the longest one may not end
// far behind the others: half of those steps, and kDirectWave for what the tiles cost
// at the least.  With 40 steps a tile for the longest instead: windows of 1 to 1e4
// points 5000 lines 164 -> 100 us, 60000 622 -> 375; one of 1e4 points in 64, 50000
// lines 460 -> 325; one of 1e5 points in 16, a line at a time 2119, by tiles 1607.
constexpr int kDirectSteps = 40, kDirectWave = 200;

struct IsoTabA {
    double mass[HK_MAX_ISO], ab[HK_MAX_ISO], ss[HK_MAX_ISO], Q[HK_MAX_ISO];
};

struct AArgs {
    const double *nu0, *S0, *EL, *A, *delta, *vy0, *nexp;
    const int32_t *iso;
    IsoTabA tab;
    int form;
    int64_t nl;
    double T, P;
    int cut_mode;
    double cut, numin, dnu;
    int64_t nx;
    const double *gK;
    double *gS, *gvy;
    double *sums;        // parts > 1: [part][4][line] sums
    double *part_tp;     // [2][block] sums over the block's lines of dL/dT, dL/dP
    int parts;
    int64_t nblocks;
};

// Line parameters and their derivatives at (T, P).
struct LineD {
    double nu, ia, S, F, y, hw, dlt;
    double dlnS_dT, dlnS_dP, dia_dT, dia_dP, dy_dT, dy_dP, dy_dvy;
};

__device__ __forceinline__ LineD line_derivs(const AArgs &a, int64_t i) {
    LineD r = {};
    const double c = kH * kC / kKB;
    const double T = a.T, P = a.P;
    const int k = a.iso ? min(max(a.iso[i], 0), HK_MAX_ISO - 1) : 0;
    const double ialphaD_h = kC * sqrt(a.tab.mass[k] / (2.0 * kKB * T));
    const bool hitran = a.form == HK_FORM_HITRAN;
    const double F0 = a.form == HK_FORM_SUPERLINE ? a.tab.ab[k] * a.tab.ss[k]
                                                  : 1.0 / a.tab.Q[k] * a.tab.ab[k] * a.tab.ss[k];
    r.dlt = hitran ? a.delta[i] : 0.0;
    r.nu = fma(r.dlt, P, a.nu0[i]);
    if (r.nu == 0.0) return r;
    r.ia = ialphaD_h / r.nu;
    const double E = a.EL[i], nu = r.nu, ia = r.ia;
    // S = S0 F with F = F0 B R ia; B, R per form (HK_FORM_*): HITRAN relative
    // to T0, ExoMol-family absolute, super-lines 1.
    const double eT = exp(-c * nu / T), e0 = exp(-c * nu / kT0);
    const double B = hitran ? exp(-E * c / T + E * c / kT0)
                            : (a.form == HK_FORM_EXOMOL ? exp(-c / T * E) : 1.0);
    const double Rr = hitran ? (1.0 - eT) / (1.0 - e0)
                             : (a.form == HK_FORM_EXOMOL ? 1.0 - eT : 1.0);
    r.F = F0 * B * Rr * ia;
    r.S = a.S0[i] * r.F;
    const double n = a.nexp[i], vy = a.vy0[i];
    const double pw = pow(kT0 / T, n);
    const double Pscale = hitran ? 1.0 / kPOatm : 1.0 / kPObar;
    const double aLp = vy * P * Pscale * pw;
    const bool super = a.form == HK_FORM_SUPERLINE;
    const double aL = aLp + (super ? 0.0 : a.A[i] / (4.0 * kPi * kC));
    r.y = aL * ia;
    r.hw = a.cut_mode == 1 ? a.cut * aL : (a.cut_mode == 2 ? a.cut / ia : a.cut);
    const double dlnR_dT = super ? 0.0 : -eT * (c * nu / (T * T)) / (1.0 - eT);
    const double dlnR_dnu = eT * (c / T) / (1.0 - eT) - e0 * (c / kT0) / (1.0 - e0);
    r.dlnS_dT = (super ? 0.0 : c * E / (T * T)) + dlnR_dT - 0.5 / T;
    r.dlnS_dP = r.dlt * (dlnR_dnu - 1.0 / nu);
    r.dia_dT = -0.5 * ia / T;
    r.dia_dP = -ia * r.dlt / nu;
    const double daL_dT = -n / T * aLp, daL_dP = vy * Pscale * pw;
    r.dy_dT = daL_dT * ia + aL * r.dia_dT;
    r.dy_dP = daL_dP * ia + aL * r.dia_dP;
    r.dy_dvy = P * Pscale * pw * ia;
    return r;
}

// Gradients of one line from its four sums; returns its dL/dT, dL/dP terms.
__device__ __forceinline__ void line_grads(const AArgs &a, const LineD &r, int64_t i, double sre,
                                           double sdy, double sdx, double sxdx, double &gT,
                                           double &gP) {
    gT = gP = 0.0;
    if (r.nu == 0.0) { a.gS[i] = 0.0; a.gvy[i] = 0.0; return; }
    a.gS[i] = r.F * sre * kISqrtPi;
    a.gvy[i] = r.S * sdy * r.dy_dvy * kISqrtPi;
    // dx/dT = d dia_dT = x dia_dT / ia (d = x_j - nu); dx/dP = -dlt ia + d dia_dP
    const double sd = sxdx / r.ia;
    const double sT = fma(sre, r.dlnS_dT, fma(sd, r.dia_dT, sdy * r.dy_dT));
    double sP = fma(sre, r.dlnS_dP, fma(sd, r.dia_dP, sdy * r.dy_dP));
    if (r.dlt != 0.0) sP = fma(-r.dlt * r.ia, sdx, sP);
    gT = r.S * sT * kISqrtPi;
    gP = r.S * sP * kISqrtPi;
}

struct WD {
    double re, dx, dy;       // Re w, dRe w/dx, dRe w/dy
};

// r2 >= 1e4: asymptotic series of w and w' (n <= 4; next terms 3e-19, 6e-18).
__device__ __forceinline__ WD wd_far(double x, double y, double r2) {
    const double inv = rcp64(r2);
    const double zr = x * inv, zi = -y * inv;
    const double ur = (zr - zi) * (zr + zi), ui = 2.0 * zr * zi;
    constexpr double c[5] = {1.0, 0.5, 0.75, 1.875, 6.5625};
    double sr = c[4], si = 0.0, tr = 9.0 * c[4], ti = 0.0;
#pragma unroll
    for (int n = 3; n >= 0; --n) {
        const double a = fma(sr, ur, fma(-si, ui, c[n]));
        si = fma(sr, ui, si * ur);
        sr = a;
        const double b = fma(tr, ur, fma(-ti, ui, (2 * n + 1) * c[n]));
        ti = fma(tr, ui, ti * ur);
        tr = b;
    }
    WD o;
    o.re = -kISqrtPi * fma(sr, zi, si * zr);
    o.dx = kISqrtPi * fma(ur, ti, ui * tr);
    o.dy = kISqrtPi * fma(ur, tr, -ui * ti);
    return o;
}

__device__ __forceinline__ WD wd_identity(double x, double y, double re, double im) {
    WD o;
    o.re = re;
    o.dx = -2.0 * fma(x, re, -y * im);
    o.dy = 2.0 * fma(x, im, y * re) - 2.0 * kISqrtPi;
    return o;
}

// 100 <= r2 < 1e4: 8-node Gauss-Hermite.
__device__ __forceinline__ WD wd_mid(double x, double y, double r2) {
    constexpr double t[4] = {kGH8t1, kGH8t2, kGH8t3, kGH8t4};
    constexpr double w[4] = {kGH8w1, kGH8w2, kGH8w3, kGH8w4};
    const double x2 = x * x;
    double sr = 0.0, si = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
        const double a = t[k] * t[k], b = t[k + 1] * t[k + 1];
        const double ua = r2 + a, ub = r2 + b;
        const double Da = fma(ua, ua, -4.0 * a * x2), Db = fma(ub, ub, -4.0 * b * x2);
        const double q = rcp64(Da * Db), ia = w[k] * (q * Db), ib = w[k + 1] * (q * Da);
        sr = fma(ua, ia, fma(ub, ib, sr));
        si = fma(r2 - a, ia, fma(r2 - b, ib, si));
    }
    return wd_identity(x, y, (2.0 / kPi) * y * sr, (2.0 / kPi) * x * si);
}

// Line core (core_value's midpoint rule, with the imaginary part): tab holds
// 1/(s^2 + y^2), tab[64 + ..] the same times s; pf = core_pole(y).
__device__ __forceinline__ WD wd_core(double x, double y, double pf, const double *tab) {
    const double ax = fmin(fabs(x), 10.0);
    const int n0 = (int)(ax * (1.0 / kHC));
    const double d = fma(-((double)n0 + 0.5), kHC, ax);
    const double *tb = tab + n0, *ts = tab + 64 + n0;
    const double r = exp_small(-2.0 * kHC * d), ri = rcp64(r);
    double P = 0.0, Q = 0.0, U = 0.0, V = 0.0;
#pragma unroll
    for (int m = kCHi; m >= 0; --m) {
        const double ce = local_const(kCE[m]);
        P = fma(P, r, ce * tb[kCHi - m]);
        U = fma(U, r, ce * ts[kCHi - m]);
        if (m > 0 && m <= kCLo) {
            Q = fma(Q, ri, ce * tb[kCHi + m]);
            V = fma(V, ri, ce * ts[kCHi + m]);
        }
    }
    const double e = (kHC / kPi) * exp_small(-d * d);
    double re = e * y * fma(Q, ri, P), im = e * fma(V, ri, U);
    if (pf != 0.0) {
        const double ex = pf * exp_neg(ax * ax), th = 2.0 * ax * y;
        re = fma(ex, cos_bounded(th), re);
        im = fma(-ex, cos_bounded(fabs(th - 0.5 * kPi)), im);      // sin
    }
    return wd_identity(x, y, re, x < 0.0 ? -im : im);
}

// 1/(s^2 + y^2) and that times s = (n0 - m + 1/2) h, for wd_core.
__device__ __forceinline__ void wd_table(double *tab, double y2) {
    const int lane = threadIdx.x & 63;
    const double s = ((double)(lane - kCHi) + 0.5) * kHC;
    wave_lds_sync();
    if (lane < kCTab) {
        const double dd = rcp64(fma(s, s, y2));
        tab[lane] = dd;
        tab[64 + lane] = s * dd;
    }
    wave_lds_sync();
}

// One line at one point per lane (on: it lies in the window), added to the
// lane's sums.  have_tab: whether tab holds this line's table yet.
__device__ __forceinline__ void add_point(bool on, double x, double y, double pf, double g,
                                          double *tab, bool &have_tab, double (&s)[4]) {
    const double y2 = y * y, r2 = fma(x, x, y2);
    WD v = {0.0, 0.0, 0.0};
    if (__ballot(on && r2 < kRB64)) {
        if (!have_tab) wd_table(tab, y2);
        have_tab = true;
        v = wd_core(x, y, pf, tab);
    }
    if (on && r2 >= kRB64) v = r2 >= kRM64 ? wd_far(x, y, r2) : wd_mid(x, y, r2);
    if (on && !(r2 >= kRB64) && !(r2 < kRB64)) v.re = v.dx = v.dy = r2;   // undefined
    if (on) {
        s[0] = fma(g, v.re, s[0]);
        s[1] = fma(g, v.dy, s[1]);
        s[2] = fma(g, v.dx, s[2]);
        s[3] = fma(g * x, v.dx, s[3]);
    }
}

// The wave's totals of s, added to lane b's sums.
__device__ __forceinline__ void add_line_totals(const double (&s)[4], int b, double (&A)[4]) {
    // rows of 16 lanes end up with s0, s2, s1, s3
    double z = swap_add16(swap_add32(s[0], s[1]), swap_add32(s[2], s[3]));
    z += row_dpp64<0xb1>(z);
    z += row_dpp64<0x4e>(z);
    z += row_dpp64<0x141>(z);
    z += row_dpp64<0x140>(z);
    const double z0 = lane_f64(z, 0), z2 = lane_f64(z, 16), z1 = lane_f64(z, 32),
                 z3 = lane_f64(z, 48);
    if ((threadIdx.x & 63) == b) { A[0] += z0; A[1] += z1; A[2] += z2; A[3] += z3; }
}

__device__ __forceinline__ int64_t lane_i64(int64_t v, int b) {
    const unsigned lo = __builtin_amdgcn_readlane((int)v, b);
    const unsigned hi = __builtin_amdgcn_readlane((int)(v >> 32), b);
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

struct AdjLDS {
    double g[kATile];
    double M0[kWaves][kFN64];                 // tile moments, one row per wave
    double Ms[kASubs][kFN64];                 // moments of the quarters
    double Mg[kASegs][kFN64];                 // and of the segments
    double G0[kFN64], Gs[kASubs][kFN64], Gg[kASegs][kFN64];
    double u[kFN64];
    double cosv[4 * kFN64];
    double tab[kWaves][128];
    double red[2][kWaves];
    int64_t range[2][kWaves];
};

// Far class: 0 near, 1: r2 in [100, 1e4) somewhere, 2: r2 >= 1e4 over the interval.
__device__ __forceinline__ int far_class_adj(double D, double half, double ia, double y) {
    const double d = fabs(D), xn = (d - half) * ia, rn = fma(xn, xn, y * y);
    const double xf = (d + half) * ia, rf = fma(xf, xf, y * y);
    return !(d >= kFarRatioAdj * half && rn >= kRB64 && rf < 1.0e30) ? 0 : rn >= kRM64 ? 2 : 1;
}

// Adds the lane's line at the interval's nodes (class cls != 0) to its sums.
__device__ __forceinline__ void add_far(int cls, double D, double half, double ia, double y,
                                        const double *G, const double *u, double (&A)[4],
                                        int k0 = 0, int k1 = kFN64) {
    const double xc = D * ia, h = half * ia;
#pragma unroll 5
    for (int k = k0; k < k1; ++k) {
        const double x = fma(u[k], h, xc), r2 = fma(x, x, y * y), g = G[k];
        const WD v = cls == 2 ? wd_far(x, y, r2) : wd_mid(x, y, r2);
        A[0] = fma(g, v.re, A[0]);
        A[1] = fma(g, v.dy, A[1]);
        A[2] = fma(g, v.dx, A[2]);
        A[3] = fma(g * x, v.dx, A[3]);
    }
}

// LPB lines per workgroup: 256, one per lane of its four waves, or 64 that all
// four waves hold, each for a quarter of the tiles' points and nodes.
// TILE points per tile (kATile at most).
template <int LPB, int TILE>
__global__ __launch_bounds__(kAT, 4) void adjoint_kernel(AArgs a) {
    __shared__ AdjLDS sh;
    constexpr int kATile = TILE, kASub = TILE / kASubs, kASegs = TILE / kASeg;
    static_assert(kASub % 64 == 0 && TILE % kAT == 0, "the tile's tables");
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t blk = blockIdx.x;
    const int part = blockIdx.y;
    constexpr bool kShared = LPB == 64;
    const int64_t i = kShared ? blk * LPB + lane : blk * LPB + t;
    if (t < 4 * kFN64) sh.cosv[t] = cos40(t);
    if (t < kFN64) sh.u[t] = node_u(t);
    LineD r = {};
    int64_t jlo = 0, jhi = 0;
    if (i < a.nl) {
        r = line_derivs(a, i);
        if (r.nu != 0.0) cut_window(r.nu, r.hw, a.numin, a.dnu, a.nx, jlo, jhi);
    }
    // tiles that some window reaches
    {
        int64_t lo = jlo < jhi ? jlo : a.nx, hi = jlo < jhi ? jhi : 0;
        for (int off = 32; off > 0; off >>= 1) {
            lo = min(lo, (int64_t)__shfl_xor((long long)lo, off, 64));
            hi = max(hi, (int64_t)__shfl_xor((long long)hi, off, 64));
        }
        if (lane == 0) { sh.range[0][wave] = lo; sh.range[1][wave] = hi; }
    }
    __syncthreads();
    int64_t lo = a.nx, hi = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        lo = min(lo, sh.range[0][w]);
        hi = max(hi, sh.range[1][w]);
    }
    const double nu = r.nu, ia = r.ia, y = r.y;
    const double pf = core_pole(y);
    double A[4] = {0.0, 0.0, 0.0, 0.0};          // sums of g times re, dy, dx, x dx
    if constexpr (kShared) {
        // windows short against the tiles they spread over: a line at a time per
        // wave, all its points, as many lines at once as the parts have waves
        double steps = (double)(jhi - jlo) * (1.0 / 64) + 1.0, most = steps;
        for (int off = 32; off > 0; off >>= 1) {
            steps += __shfl_xor(steps, off, 64);
            most = fmax(most, __shfl_xor(most, off, 64));
        }
        const int64_t rounds = (LPB + kWaves * a.parts - 1) / (kWaves * a.parts);
        const int64_t tiles = ((hi - lo) / kATile + a.parts) / a.parts;
        const double allowed = (double)(kDirectSteps * tiles);
        if (lo < hi && (double)rounds * steps <= 64.0 * allowed
            && most <= 0.5 * allowed + kDirectWave) {
            for (int b = part * kWaves + wave; b < LPB; b += kWaves * a.parts) {
                const int64_t l = lane_i64(jlo, b), h = lane_i64(jhi, b);
                const double lnu = lane_f64(nu, b), lia = lane_f64(ia, b), ly = lane_f64(y, b);
                const double lpf = lane_f64(pf, b);
                bool have_tab = false;
                double sums[4] = {0.0, 0.0, 0.0, 0.0};
                for (int64_t j0 = l; j0 < h; j0 += 64) {
                    const int64_t j = j0 + lane;
                    const bool on = j < h;
                    add_point(on, (fma((double)j, a.dnu, a.numin) - lnu) * lia, ly, lpf,
                              on ? a.gK[j] : 0.0, sh.tab[wave], have_tab, sums);
                }
                add_line_totals(sums, b, A);
            }
            hi = lo;                             // no tiles left
        }
    }
    for (int64_t tile = lo / kATile + part; lo < hi && tile <= (hi - 1) / kATile;
         tile += a.parts) {
        const int64_t j0 = tile * kATile;
        const int Wv = (int)min((int64_t)kATile, a.nx - j0);
        auto xat = [&](double p) { return fma((double)j0 + p, a.dnu, a.numin); };
        auto valid = [&](int first, int len) { return max(0, min(len, Wv - first)); };
        auto half = [&](int n) { return fmax(0.5 * (double)(n - 1), 0.5) * a.dnu; };
        auto centre = [&](int first, int n) { return xat((double)first + 0.5 * (double)max(n - 1, 0)); };
        const int wl = (int)min(max(jlo - j0, (int64_t)0), (int64_t)Wv);
        const int wh = (int)min(max(jhi - j0, (int64_t)0), (int64_t)Wv);
        const bool in = wl < wh;
        // (also the barrier behind the previous tile's readers)
        if (!__syncthreads_or(in)) continue;     // between two windows
        bool ok = true;
#pragma unroll
        for (int q = 0; q < kATile / kAT; ++q) {
            const int j = t + q * kAT;
            const double g = j < Wv ? a.gK[j0 + j] : 0.0;
            sh.g[j] = g;
            ok &= fabs(g) < 1.0e300;
        }
        for (int e = t; e < (kWaves + kASubs + kASegs) * kFN64; e += kAT) (&sh.M0[0][0])[e] = 0.0;
        // (a tile with an infinite or undefined gradient is taken point by
        // point: each line meets it at the points of its own window)
        const bool fin = __syncthreads_and(ok) != 0;
        int cls0 = 0;
        if (in && fin && wl == 0 && wh == Wv) cls0 = far_class_adj(centre(0, Wv) - nu, half(Wv), ia, y);
        const bool near = in && cls0 == 0;
        const bool any0 = __syncthreads_or(cls0) != 0, anyn = __syncthreads_or(near) != 0;
        if (any0 && valid(wave * kASub, kASub) > 0) {
            double f[kFN64];
#pragma unroll
            for (int m = 0; m < kFN64; ++m) f[m] = 0.0;
            const double xc = centre(0, Wv), ih = 1.0 / half(Wv);
            for (int q = 0; q < kASub / 64; ++q) {
                const int j = wave * kASub + q * 64 + lane;
                add_moments20(sh.g[j], (xat((double)j) - xc) * ih, f);
            }
            add_node_totals(f, sh.M0[wave]);
        }
        if (anyn && fin) {
            const int n = valid(wave * kASub, kASub);
            if (n > 0) {
                double f[kFN64];
#pragma unroll
                for (int m = 0; m < kFN64; ++m) f[m] = 0.0;
                const double xc = centre(wave * kASub, n), ih = 1.0 / half(n);
                for (int q = 0; q < kASub / 64; ++q) {
                    const int j = wave * kASub + q * 64 + lane;
                    add_moments20(sh.g[j], (xat((double)j) - xc) * ih, f);
                }
                add_node_totals(f, sh.Ms[wave]);
            }
            for (int q = 0; q < kASub / 64; ++q) {
                const int first = wave * kASub + q * 64, ns = valid(first, kASeg);
                if (ns == 0) continue;
                double f[kFN64];
#pragma unroll
                for (int m = 0; m < kFN64; ++m) f[m] = 0.0;
                add_moments20(sh.g[first + lane], (xat((double)(first + lane)) - centre(first, ns)) / half(ns), f);
                add_node_totals(f, sh.Mg[first / kASeg]);
            }
        }
        __syncthreads();
        if (any0) {
            if (t < kFN64) {
                double s = 0.0;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) s += sh.M0[w][t];
                sh.M0[0][t] = s;
            }
            if (wave == 0) {
                wave_lds_sync();
                if (lane < kFN64) sh.G0[lane] = node_weight(sh.M0[0], sh.cosv, lane);
            }
        }
        if (anyn && fin)
            for (int e = t; e < (kASubs + kASegs) * kFN64; e += kAT) {
                const int row = e / kFN64, k = e % kFN64;
                (&sh.Gs[0][0])[e] = node_weight(sh.Ms[0] + row * kFN64, sh.cosv, k);
            }
        __syncthreads();
        if (cls0)
            add_far(cls0, centre(0, Wv) - nu, half(Wv), ia, y, sh.G0, sh.u, A,
                    kShared ? wave * (kFN64 / kWaves) : 0,
                    kShared ? (wave + 1) * (kFN64 / kWaves) : kFN64);
        if (!anyn) continue;
        // quarters, then segments, then points: bit s of todo = segment s left
        unsigned todo = 0;
        for (int q = kShared ? wave : 0; q < (kShared ? wave + 1 : kASubs); ++q) {
            const int f0 = q * kASub, n = valid(f0, kASub);
            const bool inq = near && wl < f0 + n && wh > f0;
            int cls = 0;
            if (inq && fin && wl <= f0 && wh >= f0 + n)
                cls = far_class_adj(centre(f0, n) - nu, half(n), ia, y);
            if (cls) add_far(cls, centre(f0, n) - nu, half(n), ia, y, sh.Gs[q], sh.u, A);
            if (__ballot(inq && cls == 0) == 0ull) continue;
            for (int s = q * (kASub / kASeg); s < (q + 1) * (kASub / kASeg); ++s) {
                const int s0 = s * kASeg, ns = valid(s0, kASeg);
                const bool ins = inq && cls == 0 && wl < s0 + ns && wh > s0;
                int c = 0;
                if (ins && fin && wl <= s0 && wh >= s0 + ns)
                    c = far_class_adj(centre(s0, ns) - nu, half(ns), ia, y);
                if (c) add_far(c, centre(s0, ns) - nu, half(ns), ia, y, sh.Gg[s], sh.u, A);
                if (ins && c == 0) todo |= 1u << s;
            }
        }
        unsigned long long m = __ballot(todo != 0);
        double *tab = sh.tab[wave];
        while (m) {
            const int b = __builtin_ctzll(m);
            m &= m - 1ull;
            unsigned segs = __builtin_amdgcn_readlane((int)todo, b);
            const int l = __builtin_amdgcn_readlane(wl, b), h = __builtin_amdgcn_readlane(wh, b);
            const double lnu = lane_f64(nu, b), lia = lane_f64(ia, b), ly = lane_f64(y, b);
            const double lpf = lane_f64(pf, b);
            bool have_tab = false;
            double sums[4] = {0.0, 0.0, 0.0, 0.0};
            while (segs) {
                const int j = (__builtin_ctz(segs)) * kASeg + lane;
                segs &= segs - 1u;
                add_point(j >= l && j < h, (xat((double)j) - lnu) * lia, ly, lpf, sh.g[j], tab,
                          have_tab, sums);
            }
            add_line_totals(sums, b, A);
        }
    }
    bool own = i < a.nl;
    if constexpr (kShared) {
        // the four waves' sums of each line, by wave 0
        static_assert(kWaves == kASubs && sizeof(sh.g) >= sizeof(double) * kWaves * 4 * 64,
                      "one quarter per wave; sums fit the tile's gradient");
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) sh.g[(wave * 4 + q) * 64 + lane] = A[q];
        __syncthreads();
        own = own && wave == 0;
        if (own)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                A[q] = ((sh.g[q * 64 + lane] + sh.g[(4 + q) * 64 + lane]) +
                        sh.g[(8 + q) * 64 + lane]) + sh.g[(12 + q) * 64 + lane];
    }
    if (a.parts > 1) {
        if (own)
#pragma unroll
            for (int q = 0; q < 4; ++q) a.sums[((int64_t)part * 4 + q) * a.nl + i] = A[q];
        return;
    }
    double gT = 0.0, gP = 0.0;
    if (own) line_grads(a, r, i, A[0], A[1], A[2], A[3], gT, gP);
    for (int off = 32; off > 0; off >>= 1) {
        gT += __shfl_xor(gT, off, 64);
        gP += __shfl_xor(gP, off, 64);
    }
    if (lane == 0) { sh.red[0][wave] = gT; sh.red[1][wave] = gP; }
    __syncthreads();
    if (t < 2)
        a.part_tp[(int64_t)t * a.nblocks + blk] =
            ((sh.red[t][0] + sh.red[t][1]) + sh.red[t][2]) + sh.red[t][3];
}

// The parts' sums added in order, then the line's gradients (parts > 1).
__global__ __launch_bounds__(kAT) void adjoint_combine_kernel(AArgs a) {
    __shared__ double red[2][kWaves];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t i = (int64_t)blockIdx.x * kAT + t;
    double gT = 0.0, gP = 0.0;
    if (i < a.nl) {
        double A[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int p = 0; p < a.parts; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) A[q] += a.sums[((int64_t)p * 4 + q) * a.nl + i];
        line_grads(a, line_derivs(a, i), i, A[0], A[1], A[2], A[3], gT, gP);
    }
    for (int off = 32; off > 0; off >>= 1) {
        gT += __shfl_xor(gT, off, 64);
        gP += __shfl_xor(gP, off, 64);
    }
    if (lane == 0) { red[0][wave] = gT; red[1][wave] = gP; }
    __syncthreads();
    if (t < 2)
        a.part_tp[(int64_t)t * a.nblocks + blockIdx.x] =
            ((red[t][0] + red[t][1]) + red[t][2]) + red[t][3];
}

// out[r] = sum of row r of v (workgroup r; fixed order).
__global__ __launch_bounds__(1024) void sum_rows_kernel(const double *__restrict__ v, int64_t n,
                                                        double *__restrict__ out) {
    __shared__ double s[1024];
    double x = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) x += v[(int64_t)blockIdx.x * n + i];
    s[threadIdx.x] = x;
    __syncthreads();
    for (int k = 512; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// Lines per workgroup: 64 for short lists, whose 256 neighbours spread over many
// tiles, each near few of them, so that one wave went through all of a tile's
// intervals for a few lanes; and narrower tiles the fewer workgroups there are.
// Adjoint of 1000, 4000, 16000, 60000 lines with 256 lines and 1024 points 191,
// 199, 376, 756 us; with 64 lines and 1024 points 81, 102, 227, 690, with 512
// points 61, 83, 241, 653, with 256 points 43, 91, 272, 699.  2e5 lines: 1355 us
// with 256 lines, which share a tile's G_k, 1880 with 64.
constexpr int64_t kATiny = 3000;
int adjoint_lines(int64_t nlines) { return nlines < 65536 ? 64 : kAT; }

// Lists short of filling the chip several times over split each line's tiles
// over several workgroups, at most 32: up to ~20 workgroups per CU, since a
// workgroup's barriers leave its CU to the others.  3.3e5 lines, 11 tiles a
// window: 1 part 2.60 ms, 2 parts 2.28, 4 parts 2.15, 8 parts 2.32.
constexpr int kAPartBlocks = 5300, kAPartsMax = 32;
int adjoint_parts(int64_t nlines) {
    const int64_t nblocks = (nlines + adjoint_lines(nlines) - 1) / adjoint_lines(nlines);
    const int64_t p = nblocks > 0 ? kAPartBlocks / nblocks : 1;
    return (int)std::max<int64_t>(1, std::min<int64_t>(kAPartsMax, p));
}

// Workgroups whose partial dL/dT, dL/dP the last kernel adds: of the main kernel
// or, with parts, of the combination.
int64_t adjoint_sums(int64_t nlines, int parts) {
    const int per = parts > 1 ? kAT : adjoint_lines(nlines);
    return (nlines + per - 1) / per;
}

// Workspace [doubles] of a list summed in this many parts; parts == 1 needs no
// more than the two numbers a line that any caller has room for.
int64_t adjoint_doubles(int64_t nlines, int parts) {
    return 2 * adjoint_sums(nlines, parts) + (parts > 1 ? 4 * parts * nlines : 0) + 2;
}

size_t adjoint_bytes(int64_t doubles) { return (size_t)doubles * sizeof(double) + 256; }

}  // namespace

extern "C" size_t hk_voigt_adjoint_workspace_bytes(int64_t nlines) {
    if (nlines < 0) return 0;
    // enough for this list and for every shorter one in all its parts: parts *
    // lines is at most 32 lines and what adjoint_parts leaves of 5300 workgroups
    const int64_t most = (int64_t)kAPartBlocks * adjoint_lines(nlines);
    return adjoint_bytes(2 * ((nlines + 63) / 64) + 4 * std::min(kAPartsMax * nlines, most) + 2);
}

extern "C" int hk_voigt_adjoint(const hk_lines *L, const hk_tp *tp, const hk_cut *cut,
                                const hk_grid *g, const double *gK, double *gS, double *gvy,
                                double *gTP, void *ws, size_t ws_bytes, hk_stream_t stream) {
    HK_CHECK_ARG(L && tp && cut && g && gK && gS && gvy && gTP && ws,
                 "hk_voigt_adjoint: null argument");
    HK_CHECK_ARG(L->niso >= 1 && L->niso <= HK_MAX_ISO, "hk_voigt_adjoint: niso %d", L->niso);
    HK_CHECK_ARG(L->form >= HK_FORM_HITRAN && L->form <= HK_FORM_SUPERLINE,
                 "hk_voigt_adjoint: form %d", L->form);
    HK_CHECK_ARG(g->nx > 0 && g->dnu > 0.0, "hk_voigt_adjoint: bad grid");
    // in as many parts as the workspace has room for
    int parts = adjoint_parts(L->nlines);
    while (parts > 1 && ws_bytes < adjoint_bytes(adjoint_doubles(L->nlines, parts))) --parts;
    if (ws_bytes < adjoint_bytes(adjoint_doubles(L->nlines, parts))) {
        hk::set_error("hk_voigt_adjoint: workspace %zu bytes, %zu needed", ws_bytes,
                      adjoint_bytes(adjoint_doubles(L->nlines, parts)));
        return HK_ERR_WORKSPACE;
    }
    AArgs a;
    for (int k = 0; k < HK_MAX_ISO; ++k) {
        bool used = k < L->niso;
        a.tab.mass[k] = used ? L->iso_mass[k] : 1.0;
        a.tab.ab[k] = used ? L->iso_ab[k] : 0.0;
        a.tab.ss[k] = used ? L->iso_sscale[k] : 0.0;
        a.tab.Q[k] = used ? tp->Q[k] : 1.0;
    }
    a.nu0 = L->nu; a.S0 = L->S; a.EL = L->EL; a.A = L->A; a.delta = L->delta; a.vy0 = L->vy;
    a.nexp = L->n; a.iso = L->iso; a.form = L->form; a.nl = L->nlines; a.T = tp->T; a.P = tp->P;
    a.cut_mode = cut->cut_mode; a.cut = cut->cut == 0.0 ? 1.0e30 : cut->cut;
    a.numin = g->numin; a.dnu = g->dnu; a.nx = g->nx; a.gK = gK; a.gS = gS; a.gvy = gvy;
    a.parts = parts;
    a.nblocks = adjoint_sums(L->nlines, parts);
    a.part_tp = (double *)hk::align_up((size_t)ws, 256);
    a.sums = a.part_tp + 2 * a.nblocks;
    hipStream_t s = (hipStream_t)stream;
    if (a.nblocks > 0) {
        const int lines = adjoint_lines(L->nlines);
        const dim3 grid((unsigned)((L->nlines + lines - 1) / lines), (unsigned)a.parts);
        if (lines == 64 && L->nlines < kATiny)
            hipLaunchKernelGGL((adjoint_kernel<64, 256>), grid, dim3(kAT), 0, s, a);
        else if (lines == 64)
            hipLaunchKernelGGL((adjoint_kernel<64, 512>), grid, dim3(kAT), 0, s, a);
        else hipLaunchKernelGGL((adjoint_kernel<kAT, kATile>), grid, dim3(kAT), 0, s, a);
        HK_LAUNCH_CHECK();
        if (a.parts > 1) {
            hipLaunchKernelGGL(adjoint_combine_kernel, dim3((unsigned)a.nblocks), dim3(kAT), 0, s,
                               a);
            HK_LAUNCH_CHECK();
        }
    }
    hipLaunchKernelGGL(sum_rows_kernel, dim3(2), dim3(1024), 0, s, a.part_tp, a.nblocks, gTP);
    HK_LAUNCH_CHECK();
    return HK_OK;
}
