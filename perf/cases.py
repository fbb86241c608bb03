"""Timed cases of the opacity engine: the calls a user's program makes, over
the sizes it makes them with.

A case is a dict of plain values; "kind" names the call sequence:

  spectrum   line parameters at one (T, P), then the Voigt sum onto the grid
  batch      many species x (T, P): line parameters of every state, one
             prepared batched Voigt launch, the k-tables of every spectrum
  gradient   differentiable cross section, a binned loss and its backward
  profile    line parameters, then profiles with plinth removal or
             sub-Lorentzian wings
  ktable     k-table coefficients of given spectra
  kgrad      k-table coefficients and their gradient with respect to K
  products   means, k-table, reconstruction K(y) and transmission of K(y)
  sort       ordering of a raw line list on the device

The line lists follow the repository's synthetic workloads (uniform centres,
log-uniform strengths, uniform or heavy-tailed widths); sizes are those of the
workloads, of the tests and of the reference's example runs.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "helios-k_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

F64 = torch.float64
NA = 6.0221412927e23
POBAR = 0.986923                    # atm per bar
# (T, P) points of the batched workload: T 100..3000 K, P 1e-6..1e3 bar,
# paired along one path of 64
TP_PATH = 64


def listed():
    return [
        # one short window at high resolution: latency and launch count
        dict(name="spectrum_tiny_fp64", kind="spectrum", form="hitran", precision="fp64",
             lines=2000, numin=1000.0, numax=1010.0, dnu=0.001, cut_mode=0, cut=5.0,
             T=1500.0, P=1.0, niso=1, shift=False, widths="uniform"),
        # one species over the whole range in the driver's default precision:
        # 1e5 lines, 3e6 points, cut 100 (the small plain-FP64 workload)
        dict(name="spectrum_fp64", kind="spectrum", form="hitran", precision="fp64",
             lines=100000, numin=0.0, numax=30000.0, dnu=0.01, cut_mode=0, cut=100.0,
             T=1500.0, P=1.0, niso=1, shift=False, widths="uniform"),
        # a dense list on a fine grid at high pressure, FP64 (a quarter of the
        # precision-at-scale workload), four isotopologues with pressure shifts
        dict(name="spectrum_fp64_fine", kind="spectrum", form="hitran", precision="fp64",
             lines=2350001, numin=5000.0, numax=12000.0, dnu=0.001, cut_mode=0, cut=25.0,
             T=2000.0, P=10.0 * POBAR, niso=4, shift=True, widths="uniform"),
        # the precision-at-scale workload: 1e7 lines, 3e7 points, FP32C
        dict(name="spectrum_fp32c_fine", kind="spectrum", form="hitran", precision="fp32c",
             lines=10000000, numin=0.0, numax=30000.0, dnu=0.001, cut_mode=0, cut=25.0,
             T=2000.0, P=10.0 * POBAR, niso=1, shift=False, widths="uniform"),
        # an opacity table: six species of uneven size at four (T, P) of the
        # batched workload's path, with their k-tables
        dict(name="batch_fp32c", kind="batch", precision="fp32c", scale=1.0, species=6, ntp=4,
             numin=0.0, numax=30000.0, dnu=0.01, cut=100.0, nbins=300, nC=20,
             widths="uniform"),
        # retrieval: forward and backward of a binned loss (the
        # differentiation workload: a third of its 1e6 lines lies on its grid)
        dict(name="gradient", kind="gradient", lines=333333, numin=0.0, numax=10000.0,
             dnu=0.01, cut=50.0, T=1200.0, P=0.1 * POBAR, nbins=100, widths="uniform"),
        # Voigt at the 25 cm^-1 cut with the plinth removed (lines for a
        # separate continuum), a list of the size of HITRAN H2O
        dict(name="profile_plinth", kind="profile", profile=1, plinth=True, chi=False,
             lines=304225, numin=0.0, numax=30000.0, dnu=0.01, cut=25.0, T=500.0, P=1.0,
             widths="uniform"),
        # sub-Lorentzian CO2 wings around the 4.3 micron band, far cut
        dict(name="profile_sublorentz", kind="profile", profile=1, plinth=False, chi=True,
             lines=20000, numin=1800.0, numax=2800.0, dnu=0.01, cut=120.0, T=700.0, P=5.0,
             widths="uniform"),
        # k-table of one fine spectrum, bins of 1e5 points, with K(y)
        dict(name="ktable_long_bins", kind="ktable", nspec=1, nbins=300, Nxb=100000, nC=20,
             empty=0.0, want_sorted=True),
        # gradient of the k-coefficients of eight spectra on the
        # differentiation grid
        dict(name="ktable_gradient", kind="kgrad", nspec=8, nbins=100, Nxb=10000, nC=20,
             empty=0.3),
        # everything the driver derives from one spectrum after the sum
        dict(name="products", kind="products", nbins=300, Nxb=10000, nC=20, T=1500.0,
             nTr=300, dTr=0.07, empty=0.2),
        # a raw list as read from files, ordered on the device
        dict(name="sort_lines", kind="sort", lines=10000000, niso=4),
    ]


def _logu(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grid_case(rng, max_pairs, dnus, cuts, nx_lo, nx_hi, n_lo, n_hi):
    """Random grid, cut and line count with at most max_pairs line-point pairs."""
    while True:
        dnu = rng.choice(dnus)
        cut = rng.choice(cuts)
        nx = int(_logu(rng, nx_lo, nx_hi))
        if nx * dnu > 30000.0:
            continue
        numin = float(int(rng.uniform(0.0, 30000.0 - nx * dnu)))
        numax = numin + nx * dnu
        lines = int(_logu(rng, n_lo, n_hi))
        if lines * min(nx, 2.0 * cut / dnu) <= max_pairs:
            return dict(lines=lines, numin=numin, numax=numax, dnu=dnu, cut=cut)


def draw(rng):
    kind = rng.choice(["spectrum", "spectrum", "spectrum", "batch", "gradient", "profile",
                       "ktable", "kgrad", "products", "sort"])
    T = round(_logu(rng, 100.0, 3000.0), 2)
    P = float("%.4g" % _logu(rng, 1e-4, 1e2))
    widths = rng.choice(["uniform", "uniform", "heavy"])
    if kind == "spectrum":
        prec = rng.choice(["fp64", "fp64", "fp32c"])
        c = _grid_case(rng, 6e10 if prec == "fp64" else 3e11, [0.001, 0.004, 0.01, 0.05, 0.1],
                       [5.0, 25.0, 50.0, 100.0], 3e3, 1e7, 5e2, 4e6)
        c.update(kind="spectrum", form=rng.choice(["hitran", "hitran", "exomol"]), precision=prec,
                 cut_mode=0, T=T, P=P, niso=rng.choice([1, 4]), shift=rng.random() < 0.5,
                 widths=widths)
        if rng.random() < 0.2:      # cut in Lorentz half widths
            c["cut_mode"] = 1
            c["cut"] = rng.choice([40.0, 100.0])
            c["P"] = min(c["P"], 1.0)
            c["lines"] = min(c["lines"], 200000)
            c["widths"] = "uniform"
        return c
    if kind == "batch":
        return dict(kind="batch", precision="fp32c", scale=float("%.3g" % _logu(rng, 0.01, 0.6)),
                    species=rng.randint(1, 6), ntp=rng.randint(1, 6), numin=0.0, numax=30000.0,
                    dnu=rng.choice([0.01, 0.02, 0.05]), cut=rng.choice([25.0, 50.0, 100.0]),
                    nbins=rng.choice([100, 300]), nC=rng.choice([8, 20, 25]), widths=widths)
    if kind == "gradient":
        nbins = rng.choice([10, 37, 100])
        Nxb = int(_logu(rng, 2e2, 1e4))
        dnu = rng.choice([0.005, 0.01, 0.02])
        nx = nbins * Nxb
        lines = int(_logu(rng, 5e2, 5e5))
        numin = float(int(rng.uniform(100.0, 8000.0)))
        return dict(kind="gradient", lines=lines, numin=numin, numax=numin + nx * dnu, dnu=dnu,
                    cut=rng.choice([10.0, 25.0, 50.0]), T=T, P=P, nbins=nbins, widths=widths)
    if kind == "profile":
        c = _grid_case(rng, 5e8, [0.005, 0.01, 0.05], [25.0, 60.0, 120.0], 3e3, 3e6, 5e2, 3e5)
        prof = rng.choice([1, 1, 2, 3])
        c.update(kind="profile", profile=prof, plinth=rng.random() < 0.5, chi=rng.random() < 0.4,
                 T=T, P=P, widths=widths)
        return c
    if kind in ("ktable", "kgrad"):
        nC = rng.choice([8, 12, 20, 25])
        while True:
            Nxb = int(_logu(rng, 500, 2e5))
            nbins = int(_logu(rng, 1, 400))
            nspec = rng.randint(1, 8)
            if Nxb * nbins * nspec <= 1.6e7 * (1 if kind == "ktable" else 0.5) and Nxb >= 2 * nC:
                break
        c = dict(kind=kind, nspec=nspec, nbins=nbins, Nxb=Nxb, nC=nC,
                 empty=rng.choice([0.0, 0.25]))
        if kind == "ktable":
            c["want_sorted"] = rng.random() < 0.5
        return c
    if kind == "products":
        nbins = rng.choice([10, 100, 300])
        return dict(kind="products", nbins=nbins, Nxb=int(_logu(rng, 1e3, 1e4)), nC=rng.choice([12, 20]),
                    T=T, nTr=rng.choice([100, 300, 301]), dTr=rng.choice([0.05, 0.07]),
                    empty=rng.choice([0.0, 0.2]))
    return dict(kind="sort", lines=int(_logu(rng, 1e3, 8e6)), niso=rng.choice([1, 4]))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _u(g, n, lo, hi):
    return torch.rand(n, dtype=F64, device="cuda", generator=g) * (hi - lo) + lo


MASSES = (18.010565 / NA, 20.014811 / NA, 19.01478 / NA, 19.01674 / NA)
ABUNDANCE = (0.997317, 0.002, 3.72e-4, 3.11e-4)
QS = (174.58, 176.05, 1052.14, 864.74)


def _raw_lines(g, n, numin, numax, reach, widths, niso, shift, EL=2.0e4, scale=1.0):
    """An unsorted list: centres uniform over the grid and its reach (all
    positive), the repository's synthetic distributions for the rest."""
    lo = max(numin - reach, 0.01)
    d = dict(nu=_u(g, n, lo, min(numax + reach, 30000.0 + reach)))
    lg = _u(g, n, -30.0, -19.0)
    gam = _u(g, n, 0.01, 0.1)
    if widths == "heavy":
        gam = 10.0 ** _u(g, n, -4.0, 0.0)
        strong = torch.rand(n, device="cuda", generator=g) < 0.05
        lg = torch.where(strong, _u(g, n, -20.0, -17.0), lg)
    d["S"] = 10.0 ** lg * scale
    d["EL"] = _u(g, n, 0.0, EL)
    d["vy"] = gam
    d["n"] = _u(g, n, 0.3, 0.8)
    if shift:
        d["delta"] = _u(g, n, -0.01, 0.004)
    if niso > 1:
        d["iso"] = torch.randint(0, niso, (n,), dtype=torch.int32, device="cuda", generator=g)
    return d


def _iso_tables(niso):
    if niso == 1:
        return dict(iso_mass=(18.0 / NA,), iso_ab=(1.0,), iso_sscale=(1.0,)), [1.0]
    return dict(iso_mass=MASSES[:niso], iso_ab=ABUNDANCE[:niso],
                iso_sscale=(1.0,) * niso), list(QS[:niso])


FORMS = {"hitran": 0, "exomol": 1}


def _species_raw(case, seed):
    g = _gen(seed)
    form = case.get("form", "hitran")
    niso = case.get("niso", 1) if form == "hitran" else 1
    reach = case["cut"] if case.get("cut_mode", 0) == 0 else 10.0
    raw = _raw_lines(g, case["lines"], case["numin"], case["numax"], reach, case["widths"], niso,
                     case.get("shift", False) and form == "hitran")
    tab, Q = _iso_tables(niso)
    return raw, tab, Q, FORMS[form]


def _chi_of(case):
    """Perrin & Hartmann breaks and slopes at T, over the inner 80 % of the grid."""
    ab = [(0.0888, -0.160, 0.00410), (0.0, 0.0526, 0.00152), (0.0232, 0.0, 0.0)]
    w = case["numax"] - case["numin"]
    return ([3.0, 30.0, 120.0] + [a + b * math.exp(-e * case["T"]) for a, b, e in ab]
            + [case["numin"] + 0.1 * w, case["numax"] - 0.1 * w])


def _spectra(g, nspec, nbins, Nxb, empty):
    """Spectra like line sums in cm^2/g: a smooth continuum over six decades
    with narrow peaks; in half of the bins but the last a share of the points
    lies at kmin = 0 (gaps between line windows)."""
    nx = nbins * Nxb
    x = torch.linspace(0.0, 1.0, nx, dtype=F64, device="cuda")
    K = torch.empty(nspec, nx, dtype=F64, device="cuda")
    for s in range(nspec):
        lg = -1.0 + 2.0 * torch.sin(6.0 + 9.0 * s + 23.0 * x) + 1.5 * torch.sin(61.0 * x + s)
        K[s] = 10.0 ** lg
        npk = max(4, nx // 200)
        c = torch.sort(_u(g, npk, 0.0, 1.0)).values
        a = 10.0 ** _u(g, npk, -1.0, 3.0)
        w = 10.0 ** _u(g, npk, -1.0, 0.7) * 10.0 / nx
        i = torch.searchsorted(c, x).clamp(0, npk - 1)
        for k in (i, (i - 1).clamp(min=0)):
            K[s] += K[s] * a[k] / (1.0 + ((x - c[k]) / w[k]) ** 2)
        K[s] *= 1.0 + 1e-3 * torch.rand(nx, dtype=F64, device="cuda", generator=g)
    if empty > 0.0:
        gap = torch.rand(nspec, nbins, Nxb, device="cuda", generator=g) < empty
        gap &= (torch.rand(nspec, nbins, 1, device="cuda", generator=g) < 0.5)
        gap[:, -1] = False
        K.view(nspec, nbins, Nxb)[gap] = 0.0
    return K


def _batch_layout(case):
    n = [10000, 100000, 500000, 1000000, 3000000, 5000000][:case["species"]]
    m = [2.0, 16.0, 18.0, 28.0, 44.0, 48.0]
    lines = [max(200, int(v * case["scale"])) for v in n]
    tps = []
    for q in range(case["ntp"]):
        k = (q + 0.5) * (TP_PATH - 1.0) / case["ntp"]
        tps.append((100.0 * 30.0 ** (k / 63.0), 1e-6 * 10.0 ** (9.0 * k / 63.0) * POBAR))
    return lines, m, tps


def prepare(case, seed):
    from heliosk import engine as E
    kind = case["kind"]
    s = dict(case=case, E=E)
    if kind in ("spectrum", "gradient", "profile"):
        raw, tab, Q, form = _species_raw(case, seed)
        s["sp"] = E.sort_lines(**raw, **tab, form=form)
        s["Q"] = Q
        s["grid"] = E.make_grid(case["numin"], case["numax"], case["dnu"])
        if kind == "gradient":
            g = _gen(seed + 7919)
            s["T"] = torch.tensor(case["T"], dtype=F64, requires_grad=True)
            s["P"] = torch.tensor(case["P"], dtype=F64, requires_grad=True)
            s["S"] = s["sp"].S.clone().requires_grad_(True)
            s["vy"] = s["sp"].vy.clone().requires_grad_(True)
            s["w"] = _u(g, case["nbins"], 0.5, 1.5)
        else:
            s["st"] = E.State(case["lines"])
    elif kind == "batch":
        lines, masses, tps = _batch_layout(case)
        grid = E.make_grid(case["numin"], case["numax"], case["dnu"])
        g = _gen(seed)
        s["K"] = torch.empty(len(lines) * len(tps), grid.nx, dtype=F64, device="cuda")
        s["sets"], items = [], []
        for n, m in zip(lines, masses):
            raw = _raw_lines(g, n, case["numin"], case["numax"], 0.0, case["widths"], 1, False)
            sp = E.sort_lines(**raw, iso_mass=(m / NA,))
            for T, P in tps:
                st = E.line_params(sp, T, P, Q=[1.0], cut_mode=0, cut=case["cut"])
                s["sets"].append((sp, T, P, st))
                items.append((st, grid, 0.0, s["K"][len(items)]))
        mode = E.HK_VOIGT_FP32C if case["precision"] == "fp32c" else E.HK_VOIGT_FP64
        s["batch"] = E.VoigtBatch(items, mode=mode)
        s["kt"] = E.KTable(grid, case["numax"], case["nbins"], case["nC"], nspec=len(items))
    elif kind in ("ktable", "kgrad", "products"):
        g = _gen(seed)
        nspec = case.get("nspec", 1)
        s["K"] = _spectra(g, nspec, case["nbins"], case["Nxb"], case["empty"])
        nx = case["nbins"] * case["Nxb"]
        s["grid"], s["numax"] = _unit_grid(E, nx)
        s["kt"] = E.KTable(s["grid"], s["numax"], case["nbins"], case["nC"], nspec=nspec,
                           backward=kind == "kgrad")
        if kind == "kgrad":
            s["w"] = _u(g, nspec * case["nbins"] * case["nC"], -1.0, 1.0).view(
                nspec, case["nbins"], case["nC"])
            s["K"].requires_grad_(True)
    elif kind == "sort":
        g = _gen(seed)
        s["raw"] = _raw_lines(g, case["lines"], 0.0, 30000.0, 0.0, "uniform", case["niso"], True)
        s["tab"] = _iso_tables(case["niso"])[0]
    return s


def _unit_grid(E, nx):
    """A grid of nx points whose bins are whole runs of points: dnu a power
    of two, so that every grid point and bin edge is exact."""
    dnu = 2.0 ** math.floor(math.log2(30000.0 / nx))
    return E.make_grid(0.0, nx * dnu, dnu), nx * dnu


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def run(s):
    E, case = s["E"], s["case"]
    kind = case["kind"]
    if kind == "spectrum":
        st = E.line_params(s["sp"], case["T"], case["P"], Q=s["Q"], cut_mode=case["cut_mode"],
                           cut=case["cut"], state=s["st"])
        mode = E.HK_VOIGT_FP64 if case["precision"] == "fp64" else E.HK_VOIGT_FP32C
        return {"K": E.voigt(st, s["grid"], 0.0, mode)}
    if kind == "batch":
        for sp, T, P, st in s["sets"]:
            E.line_params(sp, T, P, Q=[1.0], cut_mode=0, cut=case["cut"], state=st)
        s["batch"].launch()
        coeff, nxmin = s["kt"](s["K"])
        return {"K": s["K"], "coeff": coeff, "nxmin": nxmin}
    if kind == "gradient":
        K = E.opacity(s["T"], s["P"], s["S"], s["vy"], s["sp"], s["grid"], s["Q"], 0, case["cut"])
        loss = E.binned_log_mean(K, case["nbins"], s["w"])
        gT, gP, gS, gv = torch.autograd.grad(loss, (s["T"], s["P"], s["S"], s["vy"]))
        return {"loss": loss.detach(), "gT": gT, "gP": gP, "gS": gS, "gvy": gv,
                "K": K.detach()}
    if kind == "profile":
        st = E.line_params(s["sp"], case["T"], case["P"], Q=s["Q"], cut_mode=0, cut=case["cut"],
                           state=s["st"])
        chi = _chi_of(case) if case["chi"] else None
        return {"K": E.profile(st, s["grid"], case["profile"], remove_plinth=case["plinth"],
                               chi=chi)}
    if kind == "ktable":
        out = s["kt"](s["K"], want_sorted=case["want_sorted"])
        return dict(zip(("coeff", "nxmin", "Ks"), out))
    if kind == "kgrad":
        coeff, nxmin = E.ktable_fit(s["K"], s["kt"])
        gK, = torch.autograd.grad((coeff * s["w"]).sum(), s["K"])
        return {"coeff": coeff.detach(), "nxmin": nxmin, "gK": gK}
    if kind == "products":
        K = s["K"]
        sums = E.means(K, s["grid"], case["T"])
        coeff, nxmin, Ks = s["kt"](K, want_sorted=True)
        Ky = E.ktable_reconstruct(coeff, nxmin, case["Nxb"])
        Tr = E.transmission(Ky, case["nbins"], case["Nxb"], case["nTr"], case["dTr"],
                            nxmin=nxmin.view(-1))
        return {"sums": sums, "coeff": coeff, "nxmin": nxmin, "Ks": Ks, "Ky": Ky, "Tr": Tr}
    sp = E.sort_lines(**s["raw"], **s["tab"])
    out = {k: getattr(sp, k) for k in ("nu", "S", "EL", "A", "delta", "vy", "n")}
    if sp.iso is not None:
        out["iso"] = sp.iso
    return out


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def _nx(case):
    return int((case["numax"] - case["numin"]) / case["dnu"] + 0.5)


def _core_pairs(case, T, mass_amu=18.0):
    """Points per line inside ten Doppler widths at the middle of the grid:
    no smoothness helps there, so each takes one evaluation."""
    nu = max(0.5 * (case["numin"] + case["numax"]), 1.0)
    aD = nu / 2.99792458e10 * math.sqrt(2.0 * 1.3806489e-16 * T / (mass_amu / NA))
    return max(1.0, 20.0 * aD / case["dnu"])


# floating-point operations of one profile value near the line centre, and of
# one line's smooth part (a polynomial expansion of its wings)
FLOP_CORE, FLOP_WING = 60.0, 400.0


def work(case):
    kind = case["kind"]
    if kind in ("spectrum", "profile"):
        n, nx = case["lines"], _nx(case)
        return {"bytes": 60.0 * n + 8.0 * nx,
                "flops": n * (FLOP_WING + FLOP_CORE * min(nx, _core_pairs(case, case["T"])))
                + 40.0 * nx}
    if kind == "batch":
        lines, masses, tps = _batch_layout(case)
        nx, nl = _nx(case), sum(lines)
        flops = sum(n * (FLOP_WING + FLOP_CORE * _core_pairs(case, T, m))
                    for n, m in zip(lines, masses) for T, P in tps)
        nspec = len(lines) * len(tps)
        return {"bytes": 56.0 * nl * len(tps) + nspec * (16.0 * nx + 8.0 * case["nbins"] * case["nC"]),
                "flops": flops + nspec * nx * (40.0 + 2.0 * case["nC"])}
    if kind == "gradient":
        n, nx = case["lines"], _nx(case)
        return {"bytes": 2 * 60.0 * n + 16.0 * n + 24.0 * nx,
                "flops": 3.0 * n * (FLOP_WING + FLOP_CORE * min(nx, _core_pairs(case, case["T"])))}
    if kind == "sort":
        return {"bytes": 2.0 * (56.0 + 4.0) * case["lines"], "flops": 0.0}
    pts = case.get("nspec", 1) * case["nbins"] * case["Nxb"]
    if kind == "ktable":
        return {"bytes": pts * (16.0 if case["want_sorted"] else 8.0),
                "flops": pts * (20.0 + 2.0 * case["nC"])}
    if kind == "kgrad":
        return {"bytes": pts * 24.0, "flops": pts * (40.0 + 4.0 * case["nC"])}
    return {"bytes": pts * 32.0 + 8.0 * case["nbins"] * case["nTr"],
            "flops": pts * (60.0 + 4.0 * case["nC"] + 20.0 * case["nTr"])}


# --------------------------------------------------------------------------
# The same in 64 bits from the definitions, in plain torch
# --------------------------------------------------------------------------
C_LIGHT, K_B, H_P = 2.99792458e10, 1.3806489e-16, 6.62606957e-27
ISQPI = 1.0 / math.sqrt(math.pi)
MOST_PAIRS = 8e9


def _w_trapezoid(x, y):
    """w(x + iy), y >= 0, |z| moderate: trapezoidal rule for the integral with
    the residue of the pole at z (Chiarella & Reichel 1968; Matta & Reichel
    1971), on whichever of the points kh, (k + 1/2)h lie away from x."""
    N = 14
    h = math.sqrt(math.pi / (N + 1))
    z = torch.complex(x, y)
    z2 = z * z
    f = x / h - torch.floor(x / h)
    mid = (f < 0.25) | (f > 0.75)           # x near a point kh: use the midpoints
    tot = torch.zeros_like(z)
    off = torch.where(mid, 0.5, 0.0).to(F64)
    tot = tot + torch.where(mid, torch.zeros_like(z), 0.5 / z2)
    for k in range(0, N + 2):
        t = (k + off) * h
        if k == 0:
            tot = tot + torch.where(mid, torch.exp(-t * t) / (z2 - t * t), torch.zeros_like(z))
        else:
            tot = tot + torch.exp(-t * t) / (z2 - t * t)
    w = (2j * h / math.pi) * z * tot
    q = torch.exp(torch.complex(2.0 * math.pi * y.clamp(max=math.pi / h) / h, -2.0 * math.pi * f))
    sgn = torch.where(mid, 1.0, -1.0).to(F64)
    e = torch.exp(torch.complex(y * y - x * x, -2.0 * x * y))
    pole = 2.0 * e / (1.0 + sgn * q)
    return w + torch.where(y < math.pi / h, pole, torch.zeros_like(pole))


R2_SERIES = 225.0


def _w(x, y, deriv=False):
    """w(z) and (deriv) w'(z): the asymptotic series beyond |z|^2 = 225 (13
    terms: first omitted 1e-18), the trapezoidal rule inside."""
    z = torch.complex(x, y)
    r2 = x * x + y * y
    near = r2 < R2_SERIES
    iz = 1.0 / torch.where(near, torch.full_like(z, 1e3), z)
    u = iz * iz
    cs, ds = [1.0], [1.0]
    for n in range(1, 14):
        cs.append(cs[-1] * (2 * n - 1) / 2.0)
        ds.append(cs[n] * (2 * n + 1))
    w = torch.full_like(z, cs[13])
    for n in range(12, -1, -1):
        w = w * u + cs[n]
    w = 1j * ISQPI * iz * w
    d = None
    if deriv:
        d = torch.full_like(z, ds[13])
        for n in range(12, -1, -1):
            d = d * u + ds[n]
        d = -1j * ISQPI * u * d
    idx = near.reshape(-1).nonzero().reshape(-1)
    if idx.numel():
        xs, ys = x.reshape(-1)[idx], y.expand_as(x).reshape(-1)[idx]
        ws = torch.cat([torch.where((a == 0.0) & (b == 0.0), torch.ones_like(a).to(z.dtype),
                                    _w_trapezoid(a.abs() + torch.where(a == 0.0, 1e-300, 0.0), b))
                        for a, b in zip(xs.split(1 << 22), ys.split(1 << 22))])
        ws = torch.where(xs < 0.0, ws.conj(), ws)
        w.view(-1)[idx] = ws
        if deriv:
            zs = torch.complex(xs, ys)
            d.view(-1)[idx] = -2.0 * zs * ws + 2j * ISQPI
    return (w, d) if deriv else w


def _params(case, raw, tab, Q, form):
    """Line parameters at (T, P) in 64 bits, in the sorted order of the list."""
    o = torch.argsort(raw["nu"], stable=True)
    a = {k: v[o] for k, v in raw.items()}
    T, P, T0 = case["T"], case["P"], 296.0
    c2 = H_P * C_LIGHT / K_B
    iso = a["iso"].long() if "iso" in a else torch.zeros_like(o)
    tv = lambda v: torch.tensor(list(v), dtype=F64, device="cuda")[iso]  # noqa: E731
    nu = a["nu"] + (a["delta"] * P if form == 0 and "delta" in a else 0.0)
    ia = C_LIGHT * torch.sqrt(tv(tab["iso_mass"]) / (2.0 * K_B * T)) / nu
    F = tv(tab["iso_ab"]) * tv(tab["iso_sscale"]) / tv(Q)
    eT, e0 = torch.exp(-c2 * nu / T), torch.exp(-c2 * nu / T0)
    if form == 0:
        B = torch.exp(-a["EL"] * c2 / T + a["EL"] * c2 / T0)
        F = F * B * (1.0 - eT) / (1.0 - e0) * ia
        Pn = P
    else:
        F = F * torch.exp(-c2 * a["EL"] / T) * (1.0 - eT) * ia
        Pn = P / POBAR
    pw = (T0 / T) ** a["n"]
    aL = a["vy"] * Pn * pw
    y = aL * ia
    mode = case.get("cut_mode", 0)
    hw = case["cut"] * aL if mode == 1 else case["cut"] / ia if mode == 2 else torch.full_like(nu, case["cut"])
    return dict(nu=nu, key=a["nu"], ia=ia, S=a["S"] * F, F=F, y=y, hw=hw, eT=eT, e0=e0, EL=a["EL"],
                n=a["n"], vy=a["vy"], aL=aL, pw=pw, Pn=Pn, c2=c2)


def _blocks(p, numin, dnu, nx):
    """(points, lines) blocks that hold every pair inside the cut windows."""
    reach = float((p["hw"] + (p["nu"] - p["key"]).abs()).max()) if p["nu"].numel() else 0.0
    W = 4096
    j = torch.arange(0, nx, W, device="cuda")
    lo = torch.searchsorted(p["key"], j.to(F64) * dnu + numin - reach - dnu).tolist()
    hi = torch.searchsorted(p["key"], (j + W).to(F64) * dnu + numin + reach + dnu).tolist()
    for b, (l, h) in enumerate(zip(lo, hi)):
        j0, j1 = b * W, min(nx, (b + 1) * W)
        x = torch.arange(j0, j1, device="cuda").to(F64) * dnu + numin
        for a in range(l, h, 4096):
            yield j0, j1, x, slice(a, min(h, a + 4096))


def _pairs(case):
    return case["lines"] * min(_nx(case), 2.0 * case["cut"] / case["dnu"])


def _sum_profile(case, p, profile=1, plinth=False, chi=None):
    nx = _nx(case)
    K = torch.zeros(nx, dtype=F64, device="cuda")

    def value(S, x, y):
        if profile == 1:
            return S * ISQPI * _w(x, y).real
        if profile == 2:
            return S * y / math.pi / (x * x + y * y)
        return S * ISQPI * torch.exp(-x * x)

    pl = None
    if plinth:
        pl = value(p["S"], p["hw"] * p["ia"], p["y"])
    for j0, j1, x, sl in _blocks(p, case["numin"], case["dnu"], nx):
        nu, ia, y = p["nu"][sl, None], p["ia"][sl, None], p["y"][sl, None]
        d = x[None, :] - nu
        v = value(p["S"][sl, None], d * ia, y.expand_as(d))
        if chi:
            a = d.abs()
            s1, s2, s3, b1, b2, b3, lo, hi = chi
            f = torch.exp(-b1 * (a.clamp(s1, s2) - s1) - b2 * (a.clamp(s2, s3) - s2)
                          - b3 * (a.clamp(min=s3) - s3)) * x[None, :] / nu
            v = torch.where((x > lo)[None, :] & (x < hi)[None, :], v * f, v)
        if plinth:
            v = v - pl[sl, None]
        K[j0:j1] += torch.where(d.abs() < p["hw"][sl, None], v, torch.zeros_like(v)).sum(0)
    return K


def _gradient(case, raw, tab, Q, form, w):
    p = _params(case, raw, tab, Q, form)
    nx, nb = _nx(case), case["nbins"]
    T, P = case["T"], case["P"]
    K = _sum_profile(case, p)
    m = K.view(nb, -1).mean(1)
    loss = (w * torch.log(m)).sum()
    gK = (w / m / (nx // nb)).repeat_interleave(nx // nb)
    sre, sdx, sdy = (torch.zeros_like(p["nu"]) for _ in range(3))
    for j0, j1, x, sl in _blocks(p, case["numin"], case["dnu"], nx):
        d = x[None, :] - p["nu"][sl, None]
        W, D = _w(d * p["ia"][sl, None], p["y"][sl, None].expand_as(d), deriv=True)
        g = torch.where(d.abs() < p["hw"][sl, None], gK[None, j0:j1].expand_as(d), torch.zeros_like(d))
        sre[sl] += (g * W.real).sum(1)
        sdx[sl] += (g * D.real * d).sum(1)
        sdy[sl] += (g * -D.imag).sum(1)
    c2, ia = p["c2"], p["ia"]
    dlnS = (c2 * p["EL"] / T ** 2 - p["eT"] * (c2 * p["nu"] / T ** 2) / (1.0 - p["eT"]) - 0.5 / T)
    dia = -0.5 * ia / T
    dyT = -p["n"] / T * p["aL"] * ia + p["aL"] * dia
    dyP = p["vy"] * p["pw"] * ia
    gT = (p["S"] * ISQPI * (sre * dlnS + sdx * dia + sdy * dyT)).sum()
    gP = (p["S"] * ISQPI * sdy * dyP).sum()
    gS = p["F"] * sre * ISQPI
    gv = p["S"] * sdy * (P * p["pw"] * ia) * ISQPI
    return {"loss": loss, "gT": gT, "gP": gP, "gS": gS, "gvy": gv, "K": K}


def _qr(Nxb, nC):
    """Householder QR of the Chebyshev Vandermonde matrix on Nxb points (with
    the row scaling of the reference): reflectors, their norms, diagonal."""
    x = torch.arange(Nxb, dtype=F64, device="cuda") * 2.0 / (Nxb - 1.0) - 1.0
    cols = [torch.ones_like(x), x.clone()]
    for i in range(2, nC):
        cols.append(2.0 * x * cols[-1] - cols[-2])
    V = torch.stack(cols[:nC])
    C, D = [], []
    for i in range(nC):
        v = V[i]
        v[:] = v
        scale = float(v[i:].abs().max())
        v[i:] /= scale
        s = float(v[i:].square().sum().sqrt())
        vi = float(v[i])
        sigma = -s if vi < 0.0 else s
        v[i] += sigma
        C.append(sigma * (vi + sigma))
        D.append(-scale * sigma)
        if i + 1 < nC:
            t = (V[i + 1:, i:] @ v[i:]) / C[i]
            V[i + 1:, i:] -= t[:, None] * v[None, i:]
    return V, C, D


def _fit(b, V, C, D):
    """nC - 1 reflections of b (rows) and back substitution."""
    nC = V.shape[0]
    b = b.clone()
    for j in range(nC - 1):
        t = (b[:, j:] @ V[j, j:]) / C[j]
        b[:, j:] -= t[:, None] * V[j, None, j:]
    c = torch.zeros(b.shape[0], nC, dtype=F64, device="cuda")
    c[:, nC - 1] = b[:, nC - 1] / D[nC - 1]
    for i in range(nC - 2, -1, -1):
        c[:, i] = (b[:, i] - c[:, i + 1:] @ V[i + 1:, i]) / D[i]
    return c


def _fit_t(gc, V, C, D):
    """Transpose of _fit: dL/db from dL/dc."""
    nC, Nxb = V.shape
    r = torch.zeros(gc.shape[0], Nxb, dtype=F64, device="cuda")
    a = gc.clone()
    for i in range(nC - 1):
        q = a[:, i] / D[i]
        r[:, i] = q
        a[:, i + 1:] -= q[:, None] * V[i + 1:, i][None, :]
    r[:, nC - 1] = a[:, nC - 1] / D[nC - 1]
    for j in range(nC - 2, -1, -1):
        t = (r[:, j:] @ V[j, j:]) / C[j]
        r[:, j:] -= t[:, None] * V[j, None, j:]
    return r


def _rescale(Ks, n):
    """Ks (rows: sorted bins) mapped so that its part above kmin fills the bin:
    values, left nodes and weights (identity where n = 0)."""
    Nxb = Ks.shape[1]
    k = torch.arange(Nxb, dtype=F64, device="cuda")[None, :]
    nd = n.to(F64)[:, None]
    ii = (1.0 - nd / (Nxb - 1)) * k + nd
    ii = torch.where(ii >= Nxb - 1, 0.999999 * (Nxb - 1), ii)
    il = torch.where(n[:, None] > 0, ii.long(), k.long())
    f = torch.where(n[:, None] > 0, ii - il, torch.zeros_like(ii))
    ir = (il + 1).clamp(max=Nxb - 1)
    Kl, Kr = Ks.gather(1, il), Ks.gather(1, ir)
    return Kl + (Kr - Kl) * f, il, ir, f


def _sorted_fit(K, nbins, Nxb, nC):
    Kb = K.detach().reshape(-1, Nxb)
    Ks, order = torch.sort(Kb, dim=1, stable=True)
    n = (Ks <= 0.0).sum(1)
    q = _qr(Nxb, nC)
    c = torch.cat([_fit(torch.log(_rescale(a, b)[0]), *q)
                   for a, b in zip(Ks.split(1024), n.split(1024))])
    return c, n, Ks, order, q


def _ktable_grad(case, s):
    c, n, Ks, order, q = _sorted_fit(s["K"], case["nbins"], case["Nxb"], case["nC"])
    gc = s["w"].reshape(-1, case["nC"])
    K2, il, ir, f = _rescale(Ks, n)
    gb = _fit_t(gc, *q) / K2
    gs = torch.zeros_like(Ks)
    gs.scatter_add_(1, il, gb * (1.0 - f))
    gs.scatter_add_(1, ir, gb * f)
    zero = Ks <= 0.0                 # equal values share the mean of their ranks
    tot = torch.where(zero, gs, torch.zeros_like(gs)).sum(1) / zero.sum(1).clamp(min=1)
    gs = torch.where(zero, tot[:, None].expand_as(gs), gs)
    gK = torch.empty_like(gs).scatter_(1, order, gs)
    return c, n, gK


def _reconstruct(c, n, Nxb):
    x = (-1.0 + torch.arange(Nxb, dtype=F64, device="cuda") * 2.0 / Nxb)[None, :]
    d1, d2 = torch.zeros_like(x), torch.zeros_like(x)
    for i in range(c.shape[1] - 1, 0, -1):
        d1, d2 = 2.0 * x * d1 - d2 + c[:, i, None], d1
    F = torch.exp(x * d1 - d2 + c[:, 0, None])
    k = torch.arange(Nxb, dtype=F64, device="cuda")[None, :]
    nd = n.to(F64)[:, None]
    ii = (k - nd) / (Nxb - nd - 1) * (Nxb - 1)
    ii = torch.where(ii >= Nxb - 1, 0.999999 * (Nxb - 1), ii).clamp(min=0.0)
    il = ii.long()
    Fl, Fr = F.gather(1, il), F.gather(1, il + 1)
    return torch.where(n[:, None] > 0, torch.where(k >= nd, Fl + (Fr - Fl) * (ii - il), 0.0), F)


def _transmission(Ky, n, nTr, dTr):
    Nxb = Ky.shape[1]
    m = torch.exp((torch.arange(nTr, device="cuda") - nTr // 2).to(F64) * dTr)
    w = torch.zeros(Nxb, dtype=F64, device="cuda") + 1.0
    for i, v in enumerate((-5.0 / 8.0, 1.0 / 6.0, -1.0 / 24.0)):
        w[i] += v
        w[Nxb - 3 + i] += v
    rows = []
    for b in range(Ky.shape[0]):
        a = torch.exp(-Ky[b][None, :] * m[:, None]) @ w
        nb = float(n[b])
        rows.append(a / (Nxb - 1.0) * (Nxb - nb) / Nxb + nb / Nxb)
    return torch.stack(rows)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("spectrum", "profile", "gradient"):
        if (_pairs(case) > MOST_PAIRS or case.get("cut_mode", 0) == 1):
            return None
        raw, tab, Q, form = _species_raw(case, seed)
        if kind == "gradient":
            w = _u(_gen(seed + 7919), case["nbins"], 0.5, 1.5)
            return _gradient(case, raw, tab, Q, form, w)
        p = _params(case, raw, tab, Q, form)
        if kind == "spectrum":
            return {"K": _sum_profile(case, p)}
        return {"K": _sum_profile(case, p, case["profile"], case["plinth"],
                                  _chi_of(case) if case["chi"] else None)}
    if kind == "batch":
        return None
    g = _gen(seed)
    if kind == "sort":
        raw = _raw_lines(g, case["lines"], 0.0, 30000.0, 0.0, "uniform", case["niso"], True)
        o = torch.argsort(raw["nu"], stable=True)
        out = {k: v[o] for k, v in raw.items()}
        out["A"] = torch.zeros_like(raw["nu"])
        return out
    nspec, nb, Nxb, nC = case.get("nspec", 1), case["nbins"], case["Nxb"], case["nC"]
    s = {"K": _spectra(g, nspec, nb, Nxb, case["empty"])}
    if kind == "kgrad":
        s["w"] = _u(g, nspec * nb * nC, -1.0, 1.0).view(nspec, nb, nC)
        c, n, gK = _ktable_grad(case, s)
        return {"coeff": c.view(nspec, nb, nC), "nxmin": n.view(nspec, nb).int(),
                "gK": gK.view(nspec, -1)}
    c, n, Ks, _, _ = _sorted_fit(s["K"], nb, Nxb, nC)
    out = {"coeff": c.view(nspec, nb, nC), "nxmin": n.view(nspec, nb).int()}
    if kind == "ktable":
        if case["want_sorted"]:
            out["Ks"] = Ks.view(nspec, -1)
        return out
    nx = nb * Nxb
    dnu = 2.0 ** math.floor(math.log2(30000.0 / nx))
    x = torch.arange(nx, device="cuda").to(F64) * dnu
    K = s["K"].reshape(-1)
    t1 = 2.0 * H_P * C_LIGHT ** 2 * x ** 3
    t2 = H_P * C_LIGHT / (K_B * case["T"]) * x
    B = t1 / torch.expm1(t2)
    dB = t1 * t2 / (case["T"] * 4.0 * torch.sinh(0.5 * t2.clamp(max=1400.0)) ** 2)
    B[0] = 0.0
    dB[0] = 0.0
    ros = torch.where(K != 0.0, dB / torch.where(K != 0.0, K, torch.ones_like(K)), torch.zeros_like(K))
    out["sums"] = torch.stack([(B * K).sum(), ros.sum(), B.sum(), dB.sum()])
    out["Ks"] = Ks.view(nspec, -1)
    Ky = _reconstruct(c, n, Nxb)
    out["Ky"] = Ky.reshape(-1)
    out["Tr"] = _transmission(Ky, n, case["nTr"], case["dTr"])
    return out
