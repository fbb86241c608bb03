"""Isolated lines through the far field's nodes against extended precision: the
nodes may not cost digits that the pair sum has.  Lorentz lines, and Voigt lines
so wide (y > 10) that every point lies in the wings, where the profile's own
formulas are exact to rounding.

Tolerance, relative to each point's value: a node value carries 4 roundings of
1.1e-16, interpolation at most 2.87 times that (Lebesgue constant of 20
Chebyshev nodes): 1.3e-15; its series and the Clenshaw sum, at tile and wave
level, 4 roundings: 4.4e-16; truncation 3.3e-16; the point's own formula 3e-16.
Together 2.4e-15."""
import numpy as np
import pytest

from helpers import random_lines, species_from, state_numpy

pytestmark = pytest.mark.gpu
L = np.longdouble
PI = L("3.14159265358979323846264338327950288")


def _value(profile, x, y):
    if profile == 2:
        return y / PI / (x * x + y * y)
    z = (np.abs(x) + 1j * y).astype(np.clongdouble)     # Laplace's continued fraction
    f = np.zeros_like(z)
    for n in range(90, 0, -1):
        f = (L(n) / 2) / (z - f)
    return ((1j / PI) / (z - f)).real


@pytest.mark.parametrize("nx", [20000, 600001])
@pytest.mark.parametrize("profile, P, dnu", [(2, 0.5, 0.01), (2, 0.5, 0.002), (1, 60.0, 0.05)])
@pytest.mark.parametrize("chi", [False, True])
def test_isolated_lines(nx, profile, P, dnu, chi):
    from heliosk import engine as E
    assert np.finfo(L).eps < 1e-18
    span = nx * dnu
    grid = E.make_grid(2000.0, 2000.0 + span, dnu)
    # one piece of the factor over the whole grid: exp(-B |x - nu|) x / nu
    B = 0.5 / span
    c = [0.0, 2e6, 3e6, B, B, B, 0.0, 1e9] if chi else None
    idx = np.unique(np.concatenate([np.arange(0, nx, max(1, nx // 4000)), np.arange(600)]))
    # x_j = fma(j, dnu, numin): the product in extended precision, rounded once
    x = (idx.astype(L) * L(grid.dnu) + L(grid.numin)).astype(np.float64)
    worst = 0.0
    for seed in range(12):
        d = random_lines(1, seed=seed, numin=2000.0, numax=2000.0 + span, gamma=(0.08, 0.15))
        st = E.line_params(species_from(d), 500.0, P, Q=d["iso_Q"], cut_mode=0, cut=span)
        s = state_numpy(st)
        assert profile == 2 or s["y"][0] > 10.0
        K = E.profile(st, grid, profile, chi=c).cpu().numpy()
        D = x.astype(L) - L(s["nu"][0])
        Ko = L(s["S"][0]) * _value(profile, D * L(s["ialphaD"][0]), L(s["y"][0]))
        if chi:
            Ko = Ko * np.exp(-L(B) * np.abs(D)) * (x.astype(L) / L(s["nu"][0]))
        worst = max(worst, float(np.max(np.abs(K[idx] / Ko - 1))))
    print("%.2e" % worst)
    assert worst <= 2.4e-15


@pytest.mark.parametrize("nx", [10000, 600001])
@pytest.mark.parametrize("profile, P", [(2, 0.5), (1, 60.0)])
def test_plinths_near_the_cut(nx, profile, P):
    """3000 lines close together, points near the end of their windows, where a
    line is little more than its plinth: sums of lines without their plinths,
    less a sum of plinths, would lose what the pairs' differences keep.

    Tolerance, relative to the sum with plinths: the interpolation's 2.4e-15 (the
    3000 values' own roundings, 4 * 1.1e-16 of up to 20 times the difference
    each, average out to 2e-16)."""
    from heliosk import engine as E
    dnu, cut = 100.0 / nx, 25.0
    d = random_lines(3000, seed=11, numin=2049.5, numax=2050.5, gamma=(0.08, 0.15))
    st = E.line_params(species_from(d), 500.0, P, Q=d["iso_Q"], cut_mode=0, cut=cut)
    grid = E.make_grid(2000.0, 2100.0, dnu)
    s = state_numpy(st)
    K = E.profile(st, grid, profile, remove_plinth=True).cpu().numpy()
    j = np.arange(grid.nx)
    idx = np.concatenate([j[(2000 + dnu * j > 2025.6) & (2000 + dnu * j < 2028.0)],
                          j[(2000 + dnu * j > 2072.0) & (2000 + dnu * j < 2074.4)]])
    idx = idx[:: max(1, len(idx) // 300)]
    x = (idx.astype(L) * L(grid.dnu) + L(grid.numin)).astype(np.float64)
    assert np.all(np.abs(x[:, None] - s["nu"]) < cut) and np.all(s["hw"] == cut)
    y, ia, S, nu = (s[k].astype(L) for k in ("y", "ialphaD", "S", "nu"))
    assert profile == 2 or s["y"].min() > 10.0
    pl = S * _value(profile, cut * ia, y)
    Ko = np.zeros(len(x), dtype=L)
    for i in range(3000):
        Ko += S[i] * _value(profile, (x.astype(L) - nu[i]) * ia[i], y[i]) - pl[i]
    err = float(np.max(np.abs(K[idx] / Ko - 1)))
    print("%.2e" % err)
    assert err <= 2.4e-15
