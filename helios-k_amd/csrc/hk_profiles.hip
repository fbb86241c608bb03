// hk_profiles.hip -- the line profiles other than Voigt, and plinth removal.
//
// Profiles (Line6fA_kernel<profile>, voigt.h:1235-1262, with the S1 of
// S3_kernel, voigt.h:458-470), per (line, point) pair inside the cut, in
// Doppler units x = (x_j - nu) / alpha_D and with S the line state's strength
// (S(T) / alpha_D):
//   2 Lorentz          (S y / pi) / (x^2 + y^2)
//   3 Doppler          (S / sqrt(pi)) exp(-x^2)
//   4 binned Gaussian  S / vb * (erf(x + vb/2) - erf(x - vb/2)) / 2,
//                      vb = dnu / alpha_D: the Gaussian averaged over the
//                      point's grid cell (Hill et al. 2012); the difference
//                      is formed from erfc on the side away from the centre,
//                      which keeps it accurate in the wings.
// Plinth removal (Plinth_kernel, voigt.h:1091-1164; removePlinth): every
// pair also subtracts the line's profile value at its cut, x_c = hw /
// alpha_D, so a truncated line falls to zero at the cut.  plinth_kernel forms
// the plinths of the lines once, and the sum takes them off value by value.  A
// Voigt sum with plinths is one pass in the FP64 form; in the other forms
// hk_voigt_accumulate runs first and a second pass takes the plinths off alone.
// Sub-Lorentzian wings (sLChi, voigt.h:47-72, applied at voigt.h:1345-1350 and
// in every profile branch): inside the given x range each pair's profile
// value is multiplied by chi(|x_j - nu|) x_j / nu (not the plinth); with the
// factor on, every profile -- Voigt included, through the FP64 Faddeeva
// function -- runs in this file's FP64 gather.
//
// Kernel: the FP64 tile sum of hk_voigt64.h with the profile as its parameter --
// Voigt and Lorentz wings far from a tile or a wave through Chebyshev nodes
// (with the sub-Lorentzian factor where it is one analytic piece there),
// Doppler and binned-Gaussian lines only where they do not underflow to zero,
// plinths taken off each value at nodes as at points -- so a line
// costs a few hundred evaluations, not one per point of its window.  What bounds
// it: FP64 vector instructions.  All arithmetic is FP64, in a fixed order.
// Pair by pair, Voigt with chi over 2e4 lines, 1e5 points, cut 120 took 7.0 ms,
// this 0.36; Voigt with plinth over 3e5 lines, 3e6 points, cut 25 pair by pair 3.00
// ms, a pass of the far fields and one of the plinths 1.57, in one pass 1.04.
#include <math.h>

#include "hk_device.h"
#include "hk_internal.h"
#include "hk_voigt64.h"

namespace {

using namespace hk;

__device__ __forceinline__ double prefactor(int profile, double S, double y) {
    if (profile == 2) return S * y / kPi;
    if (profile == 3 || profile == 1) return S * kISqrtPi;
    return S;
}

// Plinth of each line: its profile at the cut (0 for empty lines).
__global__ __launch_bounds__(256) void plinth_kernel(
    const double *__restrict__ S, const double *__restrict__ ia, const double *__restrict__ y,
    const double *__restrict__ hw, int64_t n, int profile, double *__restrict__ pl) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double v = 0.0;
    const double h = hw[i];
    if (h > 0.0) {
        const double xc = h * ia[i], yy = y[i];
        if (profile == 1) v = S[i] * rew64(xc, yy) * kISqrtPi;
        else if (profile == 2) v = prefactor(2, S[i], yy) / (xc * xc + yy * yy);
        else v = prefactor(3, S[i], yy) * exp(-xc * xc);
    }
    pl[i] = v;
}

struct PArgs {
    const double *nu, *S, *ia, *y, *hw, *pl, *key, *radius;
    int64_t nl;
    double numin, dnu;
    int64_t nx;
    double kmin;
    int accumulate;
    double *K;
    Chi chi;
    // sub-Lorentzian range and the points a pass writes: 0 all, 1 those inside
    // the range, -1 those outside
    double lo, hi;
    int side;
};

// PROFILE 1..4: profile sums (minus plinths when PLINTH); PROFILE 0: the
// plinth subtraction alone (after an FP32C or compat Voigt sum).
template <int PPT, int PROFILE, bool PLINTH, bool CHI, bool SPARSE>
__global__ __launch_bounds__(kThreads, 4) void profile_tiles_kernel(PArgs a) {
    __shared__ Far64LDS sh;
    if constexpr (CHI) {
        // a tile that an end of the range cuts is summed twice, as if all of it
        // lay inside and then outside: the factor is smooth over each.  (Summed
        // point by point instead, the two such tiles of a 1e5-point grid took
        // 8.1 ms, the other 96 together 1.1.)
        const int64_t j0 = (int64_t)blockIdx.x * kThreads * PPT;
        const double x0 = fma((double)j0, a.dnu, a.numin);
        const double x1 = fma((double)min(j0 + kThreads * PPT, a.nx) - 1.0, a.dnu, a.numin);
        const bool cut = (x0 <= a.lo && x1 > a.lo) || (x0 < a.hi && x1 >= a.hi);
        for (int pass = 0; pass < (cut ? 2 : 1); ++pass) {
            if (cut) {
                a.side = pass == 0 ? 1 : -1;
                a.chi.lo = pass == 0 ? -INFINITY : INFINITY;
                a.chi.hi = -a.chi.lo;
                __syncthreads();
            }
            tile_f64<PPT, LineSum<PROFILE, PLINTH, CHI, SPARSE && PROFILE <= 2 && !CHI, false, SPARSE>>(a, (int64_t)blockIdx.x, &sh);
        }
    } else {
        tile_f64<PPT, LineSum<PROFILE, PLINTH, CHI, SPARSE && PROFILE <= 2 && !CHI, false, SPARSE>>(a, (int64_t)blockIdx.x, &sh);
    }
}

template <int PROFILE, bool PLINTH, bool CHI = false>
void launch_profile(hipStream_t s, const PArgs &a) {
    constexpr bool kSparse = PROFILE != 0;      // (plinths alone are constants)
    const bool sparse = kSparse && sparse64(a.nx, a.nl);
    const int ppt = default_ppt64(a.nx, a.nl, false);
    const dim3 g((unsigned)tiles64(a.nx, ppt)), b(kThreads);
    if (sparse) {
        hipLaunchKernelGGL((profile_tiles_kernel<2, PROFILE, PLINTH, CHI, kSparse>), g, b, 0, s, a);
        return;
    }
    if (ppt == 1) hipLaunchKernelGGL((profile_tiles_kernel<1, PROFILE, PLINTH, CHI, false>), g, b, 0, s, a);
    else hipLaunchKernelGGL((profile_tiles_kernel<2, PROFILE, PLINTH, CHI, false>), g, b, 0, s, a);
}

template <int PROFILE>
void launch_chi(bool plinth, hipStream_t s, const PArgs &a) {
    if (plinth) launch_profile<PROFILE, true, true>(s, a);
    else launch_profile<PROFILE, false, true>(s, a);
}

size_t region_bytes(const hk_grid *g) {
    hk_tune t = {0, 0};
    return align_up(hk_voigt_workspace_bytes(g, &t), 256);
}

}  // namespace

extern "C" size_t hk_profile_workspace_bytes(const hk_grid *grid, int64_t nlines) {
    if (!grid || grid->nx <= 0 || nlines < 0) return 0;
    return region_bytes(grid) + align_up((size_t)nlines * sizeof(double), 256) + 512;
}

extern "C" int hk_profile_accumulate(const hk_line_state *st, const hk_grid *grid, double kmin,
                                     int accumulate, int profile, int remove_plinth,
                                     int voigt_mode, const hk_chi *chi, double *K, void *ws,
                                     size_t ws_bytes, hk_stream_t stream) {
    HK_CHECK_ARG(st && grid && K && ws, "hk_profile_accumulate: null argument");
    HK_CHECK_ARG(profile >= HK_PROFILE_VOIGT && profile <= HK_PROFILE_BINNED_GAUSS,
                 "hk_profile_accumulate: profile %d (1 Voigt, 2 Lorentz, 3 Doppler, 4 binned "
                 "Gaussian)", profile);
    HK_CHECK_ARG(!(remove_plinth && profile == HK_PROFILE_BINNED_GAUSS),
                 "hk_profile_accumulate: plinth removal is not supported for profile 4");
    HK_CHECK_ARG(grid->nx > 0 && grid->nx < ((int64_t)1 << 31) && grid->dnu > 0.0,
                 "hk_profile_accumulate: grid of %lld points, dnu %g", (long long)grid->nx,
                 grid->dnu);
    HK_CHECK_ARG(st->nlines == 0 || (st->nu && st->S && st->ialphaD && st->y && st->hw &&
                                     st->radius && st->key),
                 "hk_profile_accumulate: line state not initialised by hk_line_params");
    const size_t need = hk_profile_workspace_bytes(grid, st->nlines);
    if (ws_bytes < need) {
        set_error("hk_profile_accumulate: workspace %zu bytes, %zu needed", ws_bytes, need);
        return HK_ERR_WORKSPACE;
    }
    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)align_up((size_t)ws, 256);
    const size_t rb = region_bytes(grid);
    double *pl = (double *)(w + rb);
    if (chi) {
        HK_CHECK_ARG(chi->sigma[0] <= chi->sigma[1] && chi->sigma[1] <= chi->sigma[2],
                     "hk_profile_accumulate: chi breaks must be ascending");
    }
    // Voigt without the plinth, or in another form than FP64: the Voigt sum
    // (then the plinths alone)
    const bool voigt_sum = profile == HK_PROFILE_VOIGT && !chi &&
                           !(remove_plinth && voigt_mode == HK_VOIGT_FP64);
    if (voigt_sum) {
        hk_tune t = {0, 0};
        int rc = hk_voigt_accumulate(st, grid, kmin, accumulate, voigt_mode, &t, K, w, rb, stream);
        if (rc != HK_OK || !remove_plinth) return rc;
    }
    const int64_t n = st->nlines;
    if (remove_plinth && n > 0) {
        hipLaunchKernelGGL(plinth_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                           st->S, st->ialphaD, st->y, st->hw, n, profile, pl);
        HK_LAUNCH_CHECK();
    }
    PArgs a;
    a.nu = st->nu; a.S = st->S; a.ia = st->ialphaD; a.y = st->y; a.hw = st->hw; a.pl = pl;
    a.key = st->key; a.radius = st->radius;
    a.nl = n; a.numin = grid->numin; a.dnu = grid->dnu; a.nx = grid->nx;
    a.kmin = kmin; a.accumulate = accumulate || voigt_sum; a.K = K;
    a.chi = Chi{0, 0, 0, 0, 0, 0, 0, 0};
    a.lo = a.hi = 0.0;
    a.side = 0;
    const bool P = remove_plinth != 0;
    if (chi) {
        a.chi = Chi{chi->sigma[0], chi->sigma[1], chi->sigma[2], chi->B[0], chi->B[1], chi->B[2],
                    chi->range[0], chi->range[1]};
        a.lo = a.chi.lo;
        a.hi = a.chi.hi;
        switch (profile) {
        case HK_PROFILE_VOIGT: launch_chi<1>(P, s, a); break;
        case HK_PROFILE_LORENTZ: launch_chi<2>(P, s, a); break;
        case HK_PROFILE_DOPPLER: launch_chi<3>(P, s, a); break;
        default: launch_profile<4, false, true>(s, a); break;
        }
        HK_LAUNCH_CHECK();
        return HK_OK;
    }
    switch (profile) {
    case HK_PROFILE_VOIGT:
        voigt_sum ? launch_profile<0, true>(s, a) : launch_profile<1, true>(s, a);
        break;
    case HK_PROFILE_LORENTZ:
        P ? launch_profile<2, true>(s, a) : launch_profile<2, false>(s, a);
        break;
    case HK_PROFILE_DOPPLER:
        P ? launch_profile<3, true>(s, a) : launch_profile<3, false>(s, a);
        break;
    default: launch_profile<4, false>(s, a); break;
    }
    HK_LAUNCH_CHECK();
    return HK_OK;
}
