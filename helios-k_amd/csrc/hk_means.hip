// hk_means.hip -- consumers of the cross sections: Planck / Rosseland mean
// sums over the grid and the per-bin transmission function.
//
// Means (Mean_kernel + IntegrateMean_kernel, resample.h:635-771, called at
// heliosk.cu:1953-2000): with x_j = fma(j, dnu, numin),
//   B_j    = 2 h c^2 x^3 / (exp(h c x / (kB T)) - 1)
//   dB_j   = t1 t2 / (T (e - 2 + 1/e)),  t1 = 2 h c^2 x^3, t2 = h c x/(kB T),
//            e = exp(t2)  (dB/dT, in the form that stays finite for large t2)
//   sums   = [sum B K, sum_{K != 0} dB / K, sum B, sum dB], B = dB = 0 at x = 0.
// The reference adds a Simpson end correction inside IntegrateMean_kernel,
// but its weights (constant memory) are only set later, before the
// transmission (heliosk.cu:2392), so the means it writes are the plain sums;
// those are what is computed here.
//
// Transmission (Integrate_kernel, resample.h:541-614, heliosk.cu:2400-2440):
// for bin b of Nxb sorted values and m_t = exp((t - nTr/2) dTr),
//   a = sum_k exp(-K_k m) + sum_{i<3} (w_i exp(-K_i m) + w_{2-i} exp(-K_{Nxb-1-i} m)),
//   w = (-5/8, 1/6, -1/24),
//   Tr = a / (Nxb - 1) (Nxb - Nxmin_b) / Nxb + exp(-kmin m) Nxmin_b / Nxb.
// (The end weights are the reference's, including their order at the upper
// end.)
//
// Both are one pass over K with fixed-order reductions: deterministic.
#include <math.h>

#include "hk_device.h"
#include "hk_internal.h"
#include "hk_voigt64.h"

namespace {

constexpr int kMeanThreads = 256;
constexpr int kMeanBlocks = 1024;     // partial sums per launch (fixed order)

__device__ inline void planck_terms(double x, double T, double &B, double &dB) {
    using namespace hk;
    const double t1 = 2.0 * kH * x * x * x * kC * kC;
    const double t2 = kH * x * kC / (kKB * T);
    const double e = exp(t2);
    B = t1 / (e - 1.0);
    dB = t1 * t2 / (T * (e - 2.0 + 1.0 / e));
    if (x == 0.0) { B = 0.0; dB = 0.0; }
}

// Per block: the four sums over points j = block*256 + tid + k*stride.
__global__ __launch_bounds__(kMeanThreads) void means_partial_kernel(
    const double *__restrict__ K, double numin, double dnu, int64_t nx, double T,
    double *__restrict__ part) {
    __shared__ double s[4][kMeanThreads];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kMeanThreads;
    for (int64_t j = (int64_t)blockIdx.x * kMeanThreads + threadIdx.x; j < nx; j += stride) {
        double B, dB;
        planck_terms(fma((double)j, dnu, numin), T, B, dB);
        const double k = K[j];
        a0 += B * k;
        if (k != 0.0) a1 += dB / k;
        a2 += B;
        a3 += dB;
    }
    const int t = threadIdx.x;
    s[0][t] = a0; s[1][t] = a1; s[2][t] = a2; s[3][t] = a3;
    __syncthreads();
    for (int h = kMeanThreads / 2; h > 0; h >>= 1) {
        if (t < h)
            for (int q = 0; q < 4; ++q) s[q][t] += s[q][t + h];
        __syncthreads();
    }
    if (t < 4) part[(size_t)blockIdx.x * 4 + t] = s[t][0];
}

// Trapezoid form on explicit points x (IntegrateMean_kernel with
// useIndividualX, resample.h:700-716): per interval [x_j, x_j+1] the mean of
// the end values times the width; the Rosseland term needs both K != 0.
__global__ __launch_bounds__(kMeanThreads) void means_x_partial_kernel(
    const double *__restrict__ K, const double *__restrict__ x, int64_t nx, double T,
    double *__restrict__ part) {
    __shared__ double s[4][kMeanThreads];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kMeanThreads;
    for (int64_t j = (int64_t)blockIdx.x * kMeanThreads + threadIdx.x; j + 1 < nx; j += stride) {
        double B0, dB0, B1, dB1;
        const double x0 = x[j], x1 = x[j + 1];
        planck_terms(x0, T, B0, dB0);
        planck_terms(x1, T, B1, dB1);
        const double k0 = K[j], k1 = K[j + 1], w = x1 - x0;
        a0 += 0.5 * (B0 * k0 + B1 * k1) * w;
        if (k0 != 0.0 && k1 != 0.0) a1 += 0.5 * (dB0 / k0 + dB1 / k1) * w;
        a2 += 0.5 * (B0 + B1) * w;
        a3 += 0.5 * (dB0 + dB1) * w;
    }
    const int t = threadIdx.x;
    s[0][t] = a0; s[1][t] = a1; s[2][t] = a2; s[3][t] = a3;
    __syncthreads();
    for (int h = kMeanThreads / 2; h > 0; h >>= 1) {
        if (t < h)
            for (int q = 0; q < 4; ++q) s[q][t] += s[q][t + h];
        __syncthreads();
    }
    if (t < 4) part[(size_t)blockIdx.x * 4 + t] = s[t][0];
}

__global__ __launch_bounds__(kMeanThreads) void means_final_kernel(
    const double *__restrict__ part, int nblocks, double *__restrict__ sums) {
    __shared__ double s[4][kMeanThreads];
    const int t = threadIdx.x;
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = t; b < nblocks; b += kMeanThreads)
        for (int q = 0; q < 4; ++q) a[q] += part[(size_t)b * 4 + q];
    for (int q = 0; q < 4; ++q) s[q][t] = a[q];
    __syncthreads();
    for (int h = kMeanThreads / 2; h > 0; h >>= 1) {
        if (t < h)
            for (int q = 0; q < 4; ++q) s[q][t] += s[q][t + h];
        __syncthreads();
    }
    if (t < 4) sums[t] = s[t][0];
}

constexpr int kTrDThreads = 256;
constexpr int kTrM = 8;               // m values per workgroup

// grid (ceil(nTr / kTrM), nbins): one workgroup sums kTrM transmission
// points of one bin; K of the bin is read once per workgroup (coalesced).
__global__ __launch_bounds__(kTrDThreads) void transmission_direct_kernel(
    const double *__restrict__ Ks, int Nxb, const int32_t *__restrict__ nxmin, double kmin,
    int nTr, double dTr, double *__restrict__ Tr) {
    __shared__ double s[kTrM][kTrDThreads];
    const int b = blockIdx.y;
    const int t0 = blockIdx.x * kTrM;
    const int tid = threadIdx.x;
    const double *Kb = Ks + (size_t)b * Nxb;
    double m[kTrM], a[kTrM];
#pragma unroll
    for (int q = 0; q < kTrM; ++q) {
        m[q] = exp((double)(t0 + q - nTr / 2) * dTr);
        a[q] = 0.0;
    }
    for (int k = tid; k < Nxb; k += kTrDThreads) {
        const double kv = Kb[k];
#pragma unroll
        for (int q = 0; q < kTrM; ++q) a[q] += exp(-kv * m[q]);
    }
    if (tid < 3) {
        const double w[3] = {-5.0 / 8.0, 1.0 / 6.0, -1.0 / 24.0};
        const double klo = Kb[tid], khi = Kb[Nxb - 1 - tid];
#pragma unroll
        for (int q = 0; q < kTrM; ++q) {
            a[q] += w[tid] * exp(-klo * m[q]);
            a[q] += w[2 - tid] * exp(-khi * m[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < kTrM; ++q) s[q][tid] = a[q];
    __syncthreads();
    for (int h = kTrDThreads / 2; h > 0; h >>= 1) {
        if (tid < h)
#pragma unroll
            for (int q = 0; q < kTrM; ++q) s[q][tid] += s[q][tid + h];
        __syncthreads();
    }
    if (tid < kTrM && t0 + tid < nTr) {
        const double nmin = nxmin ? (double)nxmin[b] : 0.0;
        const double nb = (double)Nxb;
        Tr[(size_t)b * nTr + t0 + tid] =
            s[tid][0] / (nb - 1.0) * (nb - nmin) / nb + exp(-kmin * m[tid]) * nmin / nb;
    }
}

constexpr int kTrThreads = 512;
constexpr int kTrWaves = kTrThreads / 64;
constexpr int kTrPer = kTrWaves * 16;        // m values per workgroup, 16 a wave
constexpr int kTrC = 128;                    // points per cluster
constexpr int kTrBatch = 128;                // clusters in LDS at a time
constexpr int kTrSuper = 16;                 // clusters per super-cluster
// Largest half width of a cluster times m that its nodes may stand for: 20
// Chebyshev nodes leave 2 I_20(3) = 2e-15 of e^{-K m} at the cluster's least K.
constexpr double kTrNodes = 3.0;
// e^-t is 0 from t = 745.2 on.
constexpr double kTrZero = 746.0;
// A cluster whose terms are all below e^-50 of the bin's largest adds less than
// a rounding (1e-18 of the sum for 1e4 points).
constexpr double kTrNone = 50.0;

// e^-t (t clamped where the result is 0 or infinite).
__device__ __forceinline__ double tr_exp(double t) {
    t = t > 800.0 ? 800.0 : t;
    return hk::exp_neg(t < -800.0 ? -800.0 : t);
}

// Minimum of v over the wave, in every lane.
__device__ __forceinline__ double wave_min64(double v) {
    v = fmin(v, hk::row_dpp64<0xb1>(v));
    v = fmin(v, hk::row_dpp64<0x4e>(v));
    v = fmin(v, hk::row_dpp64<0x141>(v));
    v = fmin(v, hk::row_dpp64<0x140>(v));
    return fmin(fmin(hk::lane_f64(v, 0), hk::lane_f64(v, 16)),
                fmin(hk::lane_f64(v, 32), hk::lane_f64(v, 48)));
}

// Whether nodes may stand for a cluster of this half width: 1 / half is finite
// (subnormal spans, e.g. of tails that underflow, are summed value by value).
__device__ __forceinline__ bool tr_half_ok(double half) { return !(half > 0.0 && half < 1.0e-290); }

// Place in [-1, 1] of a value that lies d above the cluster's least.  From the
// difference, not from a midpoint: that of two neighbouring doubles rounds onto
// one of them, and T_19 of a place of +-2 is 4e10.
__device__ __forceinline__ double tr_place(double d, double half, double ih) {
    return fmin(fmax((d - half) * ih, -1.0), 1.0);
}

struct TrCluster {
    double lo, half;
    int n, nodes;            // points; whether the nodes may stand for them
};

// One workgroup sums up to kTrPer transmission points of one bin.  The bin is
// taken in clusters of kTrC consecutive values: e^{-K m} is entire in K, so over
// a cluster whose half width h has h m <= 3 the sum over its values is that over
// 20 Chebyshev nodes with the values' Lagrange weights, whatever m; a cluster
// too wide for an m is summed value by value, and one with nothing left to add
// is skipped.  Sixteen clusters make a super-cluster, whose nodes stand for them
// where they are narrow enough for the m.  The waves make the clusters of a batch
// together, then each takes its 16 m values, four lanes each, without waiting for
// the others.  A cluster's range is its values' own, so bins that are not sorted
// are summed too, more slowly.
// Bound by FP64 vector instructions (300 bins of 1e4 points, 300 m: one
// exponential per point and m takes 633 us, this 256).
__global__ __launch_bounds__(kTrThreads, 4) void transmission_kernel(
    const double *__restrict__ Ks, int Nxb, const int32_t *__restrict__ nxmin, double kmin,
    int nTr, double dTr, double *__restrict__ Tr) {
    using namespace hk;
    __shared__ double Gp[kFN64 / 4][kTrBatch][4];     // node weights, node 4k + part
    __shared__ double Mw[kTrWaves][3 * kFN64];
    __shared__ TrCluster cl[kTrBatch], sc[kTrBatch / kTrSuper];
    __shared__ double Gs[kTrBatch / kTrSuper][kFN64];
    __shared__ double cosv[4 * kFN64];
    __shared__ double red[kTrWaves];
    const int b = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, part = tid & 3;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double *Kb = Ks + (size_t)b * Nxb;
    // four lanes per m; a wave past the last has none
    const int ti = blockIdx.x * kTrPer + 16 * wave + (lane >> 2);
    const bool any_m = blockIdx.x * kTrPer + 16 * wave < nTr;
    const double m = exp((double)(ti - nTr / 2) * dTr);
    if (tid < 4 * kFN64) cosv[tid] = cos40(tid);
    double least = INFINITY;
    for (int k = tid; k < Nxb; k += kTrThreads) least = fmin(least, Kb[k]);
    least = wave_min64(least);
    if (lane == 0) red[wave] = least;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kTrWaves; ++w) least = fmin(least, red[w]);
    double a = 0.0;
    double un[kFN64 / 4];                  // (K - lo) / half at this lane's nodes
#pragma unroll
    for (int k = 0; k < kFN64 / 4; ++k)
        un[k] = 1.0 + node_u(4 * k + part);
    for (int k0 = 0; k0 < Nxb; k0 += kTrC * kTrBatch) {
        const int ncl = min(kTrBatch, (Nxb - k0 + kTrC - 1) / kTrC);
        __syncthreads();                    // the previous batch's readers are done
        // three at a time: their node weights come from 60 lanes together
        for (int c3 = wave * 3; c3 < ncl; c3 += kTrWaves * 3) {
            double *M = Mw[wave];
            wave_lds_sync();
            if (lane < 3 * kFN64) M[lane] = 0.0;
            wave_lds_sync();
            for (int c = c3; c < min(c3 + 3, ncl); ++c) {
                // range and moments
                const int first = k0 + c * kTrC, n = min(kTrC, Nxb - first);
                double v[kTrC / 64];
                double lo = INFINITY, hi = -INFINITY;
                bool fin = true;
#pragma unroll
                for (int q = 0; q < kTrC / 64; ++q) {
                    const int k = lane + 64 * q;
                    v[q] = k < n ? Kb[first + k] : 0.0;
                    if (k < n) {
                        lo = fmin(lo, v[q]);
                        hi = fmax(hi, v[q]);
                        fin &= fabs(v[q]) < 1.0e300;
                    }
                }
                lo = wave_min64(lo);
                hi = -wave_min64(-hi);
                const double half = 0.5 * (hi - lo);
                const bool nodes = __ballot(!fin) == 0ull && tr_half_ok(half);
                if (nodes) {
                    double f[kFN64];
#pragma unroll
                    for (int q = 0; q < kFN64; ++q) f[q] = 0.0;
                    const double ih = half > 0.0 ? 1.0 / half : 0.0;
#pragma unroll
                    for (int q = 0; q < kTrC / 64; ++q)
                        add_moments20(lane + 64 * q < n ? 1.0 : 0.0, tr_place(v[q] - lo, half, ih),
                                      f);
                    add_node_totals(f, M + (c - c3) * kFN64);
                }
                // (without nodes -- undefined or infinite values -- never skipped)
                if (lane == 0) cl[c] = TrCluster{nodes ? lo : -INFINITY, half, n, nodes ? 1 : 0};
            }
            wave_lds_sync();
            const int c = c3 + lane / kFN64, k = lane % kFN64;
            if (lane < 3 * kFN64 && c < ncl)
                Gp[k >> 2][c][k & 3] = node_weight(M + lane / kFN64 * kFN64, cosv, k);
        }
        __syncthreads();
        // super-clusters, from the nodes of their clusters
        const int nsc = (ncl + kTrSuper - 1) / kTrSuper;
        for (int h = wave; h < nsc; h += kTrWaves) {
            const int c0 = h * kTrSuper, nc = min(kTrSuper, ncl - c0);
            double lo = INFINITY, span = 0.0;
            int ok = 1;
            for (int c = c0; c < c0 + nc; ++c) {
                lo = fmin(lo, cl[c].lo);
                ok &= cl[c].nodes;
            }
            for (int c = c0; c < c0 + nc; ++c)
                span = fmax(span, fma(2.0, cl[c].half, cl[c].lo - lo));
            const double half = 0.5 * span;
            ok &= tr_half_ok(half);
            if (ok) {
                double f[kFN64];
#pragma unroll
                for (int q = 0; q < kFN64; ++q) f[q] = 0.0;
                const double ih = half > 0.0 ? 1.0 / half : 0.0;
                for (int q = lane; q < kTrSuper * kFN64; q += 64) {
                    const int c = c0 + min(q / kFN64, nc - 1), k = q % kFN64;
                    const double K = fma(cl[c].half, 1.0 + cosv[2 * k + 1], cl[c].lo - lo);
                    add_moments20(q / kFN64 < nc ? Gp[k >> 2][c][k & 3] : 0.0,
                                  tr_place(K, half, ih), f);
                }
                double *M = Mw[wave];
                wave_lds_sync();
                if (lane < kFN64) M[lane] = 0.0;
                wave_lds_sync();
                add_node_totals(f, M);
                wave_lds_sync();
                if (lane < kFN64) Gs[h][lane] = node_weight(M, cosv, lane);
            }
            if (lane == 0) sc[h] = TrCluster{lo, half, 0, ok};
        }
        __syncthreads();
        if (any_m) {
            // e^{-lo m} (the product's rounding, eps lo m of the value, put
            // back) times the nodes' e^{-(K - lo) m}, argument <= 6
            auto by_nodes = [&](const TrCluster &q, const double (&w)[kFN64 / 4]) {
                const double hm = fmin(q.half * m, kTrNodes);
                double v = 0.0;
#pragma unroll
                for (int k = 0; k < kFN64 / 4; ++k) v = fma(w[k], exp_neg(un[k] * hm), v);
                const double p = q.lo * m, e = fma(q.lo, m, -p);
                return v * (tr_exp(p) * (1.0 - e));
            };
            auto none = [&](const TrCluster &q) {
                return (q.lo - least) * m > kTrNone || q.lo * m > kTrZero;
            };
            double w[kFN64 / 4];
            for (int h = 0; h < nsc; ++h) {
                const TrCluster s = sc[h];
                const bool off = none(s), whole = s.nodes && s.half * m <= kTrNodes;
                if (__ballot(!off && whole) != 0ull) {
#pragma unroll
                    for (int k = 0; k < kFN64 / 4; ++k) w[k] = Gs[h][4 * k + part];
                    const double v = by_nodes(s, w);
                    a += !off && whole ? v : 0.0;
                }
                const bool rest = !off && !whole;
                if (__ballot(rest) == 0ull) continue;
                for (int c = h * kTrSuper; c < min(ncl, (h + 1) * kTrSuper); ++c) {
                    const TrCluster q = cl[c];
                    const bool in = rest && !none(q), nodes = q.nodes && q.half * m <= kTrNodes;
                    if (__ballot(in && nodes) != 0ull) {
#pragma unroll
                        for (int k = 0; k < kFN64 / 4; ++k) w[k] = Gp[k][c][part];
                        const double v = by_nodes(q, w);
                        a += in && nodes ? v : 0.0;
                    }
                    if (__ballot(in && !nodes) != 0ull) {
                        const double *Kc = Kb + k0 + c * kTrC;
                        double v[kTrC / 64];
#pragma unroll
                        for (int i = 0; i < kTrC / 64; ++i)
                            v[i] = lane + 64 * i < q.n ? Kc[lane + 64 * i] : INFINITY;
                        double t = 0.0;
#pragma unroll
                        for (int i = 0; i < kTrC / 64; ++i)
                            for (int k = part; k < 64; k += 4) {
                                const double kv = __shfl(v[i], k, 64);
                                t += kv < INFINITY || !(kv == kv) ? tr_exp(kv * m) : 0.0;
                            }
                        a += in && !nodes ? t : 0.0;
                    }
                }
            }
        }
    }
    if (!any_m) return;
    const double nmin = nxmin ? (double)nxmin[b] : 0.0, nb = (double)Nxb;
    if (part < 3) {                         // Simpson end weights, a term per lane
        const double w[3] = {-5.0 / 8.0, 1.0 / 6.0, -1.0 / 24.0};
        a = fma(part == 0 ? w[0] : part == 1 ? w[1] : w[2], tr_exp(Kb[part] * m), a);
        a = fma(part == 0 ? w[2] : part == 1 ? w[1] : w[0], tr_exp(Kb[Nxb - 1 - part] * m), a);
    }
    a += __shfl_xor(a, 1, 64);
    a += __shfl_xor(a, 2, 64);
    if (part == 0 && ti < nTr)
        Tr[(size_t)b * nTr + ti] =
            a / (nb - 1.0) * (nb - nmin) / nb + exp(-kmin * m) * nmin / nb;
}

// Whether the clusters take a transmission, else every value is exponentiated.
// Measured: the direct kernel adds 1.24e6 to 1.42e6 terms per us, by the values,
// once it fills the chip; a workgroup of the clusters, 512 of which run at once,
// takes 60 us and 5.5 us per 1000 points, little of which others can hide; they
// have to be a fifth faster by this.  300 bins of 1e4 points, 300 m: 633 us direct,
// 256 clusters; 80 bins 178 and 126; 300 of 1714: 136 and 141; 10 of 9059: 37 and
// 110.
bool transmission_by_clusters(int nbins, int Nxb, int nTr) {
    const double direct = (double)nbins * Nxb * nTr / 1.24e6;
    const double blocks = (double)nbins * ((nTr + kTrPer - 1) / kTrPer);
    return direct > 1.2 * (60.0 + 0.0055 * Nxb) * fmax(1.0, blocks / 512.0);
}

}  // namespace

extern "C" size_t hk_means_workspace_bytes(void) {
    return (size_t)kMeanBlocks * 4 * sizeof(double) + 256;
}

extern "C" int hk_means(const double *K, const hk_grid *grid, double T, double *sums,
                        void *workspace, size_t workspace_bytes, hk_stream_t stream) {
    HK_CHECK_ARG(K && grid && sums && workspace, "hk_means: null argument");
    HK_CHECK_ARG(grid->nx > 0 && grid->dnu > 0.0, "hk_means: empty grid or dnu <= 0");
    HK_CHECK_ARG(T > 0.0, "hk_means: T must be > 0");
    if (workspace_bytes < hk_means_workspace_bytes()) {
        hk::set_error("hk_means: workspace %zu bytes, %zu needed", workspace_bytes,
                      hk_means_workspace_bytes());
        return HK_ERR_WORKSPACE;
    }
    double *part = (double *)hk::align_up((size_t)workspace, 256);
    const int64_t want = (grid->nx + kMeanThreads - 1) / kMeanThreads;
    const int nblocks = (int)(want < kMeanBlocks ? want : kMeanBlocks);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(means_partial_kernel, dim3(nblocks), dim3(kMeanThreads), 0, s, K,
                       grid->numin, grid->dnu, grid->nx, T, part);
    HK_LAUNCH_CHECK();
    hipLaunchKernelGGL(means_final_kernel, dim3(1), dim3(kMeanThreads), 0, s, part, nblocks,
                       sums);
    HK_LAUNCH_CHECK();
    return HK_OK;
}

extern "C" int hk_means_x(const double *K, const double *x, int64_t nx, double T, double *sums,
                          void *workspace, size_t workspace_bytes, hk_stream_t stream) {
    HK_CHECK_ARG(K && x && sums && workspace, "hk_means_x: null argument");
    HK_CHECK_ARG(nx > 0, "hk_means_x: no points");
    HK_CHECK_ARG(T > 0.0, "hk_means_x: T must be > 0");
    if (workspace_bytes < hk_means_workspace_bytes()) {
        hk::set_error("hk_means_x: workspace %zu bytes, %zu needed", workspace_bytes,
                      hk_means_workspace_bytes());
        return HK_ERR_WORKSPACE;
    }
    double *part = (double *)hk::align_up((size_t)workspace, 256);
    const int64_t want = (nx + kMeanThreads - 1) / kMeanThreads;
    const int nblocks = (int)(want < kMeanBlocks ? want : kMeanBlocks);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(means_x_partial_kernel, dim3(nblocks), dim3(kMeanThreads), 0, s, K, x, nx, T,
                       part);
    HK_LAUNCH_CHECK();
    hipLaunchKernelGGL(means_final_kernel, dim3(1), dim3(kMeanThreads), 0, s, part, nblocks,
                       sums);
    HK_LAUNCH_CHECK();
    return HK_OK;
}

extern "C" int hk_transmission(const double *Ksorted, int nbins, int Nxb, const int32_t *nxmin,
                               double kmin, int nTr, double dTr, double *Tr,
                               hk_stream_t stream) {
    HK_CHECK_ARG(Ksorted && Tr, "hk_transmission: null argument");
    HK_CHECK_ARG(nbins > 0 && nbins <= 65535, "hk_transmission: nbins %d out of 1..65535", nbins);
    HK_CHECK_ARG(Nxb >= 3, "hk_transmission: %d points per bin (at least 3)", Nxb);
    HK_CHECK_ARG(nTr > 0, "hk_transmission: nTr must be > 0");
    hipStream_t s = (hipStream_t)stream;
    if (transmission_by_clusters(nbins, Nxb, nTr)) {
        dim3 g((unsigned)((nTr + kTrPer - 1) / kTrPer), (unsigned)nbins);
        hipLaunchKernelGGL(transmission_kernel, g, dim3(kTrThreads), 0, s, Ksorted, Nxb, nxmin,
                           kmin, nTr, dTr, Tr);
    } else {
        dim3 g((unsigned)((nTr + kTrM - 1) / kTrM), (unsigned)nbins);
        hipLaunchKernelGGL(transmission_direct_kernel, g, dim3(kTrDThreads), 0, s, Ksorted, Nxb,
                           nxmin, kmin, nTr, dTr, Tr);
    }
    HK_LAUNCH_CHECK();
    return HK_OK;
}
